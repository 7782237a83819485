"""What the compiler reports about the built kernels: a prompt kernel whose operands land in scratch waits for memory inside its main loop."""
import os
import re
import struct
import subprocess

import pytest

from ktransformers_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib):
    """The gfx950 code objects of a library."""
    data = open(lib, "rb").read()
    for m in re.finditer(MAGIC, data):
        at = m.start()
        pos, (n,) = at + 32, struct.unpack_from("<Q", data, at + 24)
        for _ in range(n):
            ofs, size, idlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if size and b"gfx950" in triple:
                yield data[at + ofs:at + ofs + size]


def private_segments(lib, tmp):
    """{mangled kernel name: bytes of scratch per lane} over the gfx950 code objects of a library."""
    out = {}
    for code in code_objects(lib):
        tmp.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(tmp)], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n\s+- \.", notes):
            name, priv = re.search(r"\.?name:\s+(_Z\S+)", k), re.search(r"private_segment_fixed_size:\s+(\d+)", k)
            if name and priv:
                out[name.group(1)] = int(priv.group(1))
    return out


@pytest.mark.parametrize("kernel", ["moe_gguf_fold_kernel", "moe_rawint4_chunk_kernel", "mla_decode_wide_kernel", "lin_tile_kernel", "moe_gemm_stream_kernel", "moe_fp8_stream_kernel", "mla_prefill_kernelILb1E", "mla_prefill_kernelILb0ELb1E"])
def test_prompt_kernels_keep_their_operands_in_registers(kernel, tmp_path):
    if not os.path.exists(build.LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    seen = {k: v for k, v in private_segments(build.LIB, tmp_path / "code.o").items() if kernel in k}
    assert seen, f"{kernel}: not in {build.LIB}"
    assert not {k: v for k, v in seen.items() if v}, "scratch bytes per lane"


def undrained(lines):
    """LDS-DMA requests of a kernel's listing from which a path leads to the kernel's end without a wait for all of them."""
    code, at = [], {}
    for line in lines:
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+): ", line)
        if m:
            target = re.search(r"<\S+\+0x([0-9a-f]+)>\s*$", line)
            at[int(m.group(3), 16)] = len(code)
            code.append((m.group(1), m.group(2), int(target.group(1), 16) if target else 0))
    start = min(at)

    def after(i):
        op, _, target = code[i]
        if op == "s_endpgm":
            return []
        jump = [at[start + target]] if op == "s_branch" or op.startswith("s_cbranch") else []
        return jump if op == "s_branch" else jump + [i + 1]

    bad, requests = [], [i for i, c in enumerate(code) if re.match(r"(global_load_lds|buffer_load)", c[0]) and ("lds" in c[0] or "lds" in c[1])]
    for r in requests:
        todo, seen = after(r), set()
        while todo:
            i = todo.pop()
            if i in seen or (code[i][0] == "s_waitcnt" and "vmcnt(0)" in code[i][1]):
                continue
            seen.add(i)
            if code[i][0] == "s_endpgm":
                bad.append(r)
                break
            todo += after(i)
    return bad, len(requests)


@pytest.mark.parametrize("kernel", ["moe_rawint4_chunk_kernel", "moe_gemm_stream_kernel", "moe_fp8_stream_kernel", "mla_prefill_kernelILb1E"])
def test_no_request_outlives_its_workgroup(kernel, tmp_path):
    """A workgroup's LDS goes to the next one when it ends: every path from a request that writes there passes a wait for all requests."""
    if not os.path.exists(build.LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    seen = 0
    for code in code_objects(build.LIB):
        if kernel.encode() not in code:
            continue
        (tmp_path / "code.o").write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", str(tmp_path / "code.o")], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
            if kernel in part.split("\n", 1)[0]:
                bad, requests = undrained(part.split("\n")[1:])
                assert requests and not bad, f"{part.split(chr(10), 1)[0]}: {len(bad)} of {requests} requests may outlive the workgroup"
                seen += 1
    assert seen, f"{kernel}: not in {build.LIB}"


def test_scales_are_read_behind_a_wait_for_them(tmp_path):
    """lin_tile_kernel's FP8 weight scales come by LDS-DMA, which the compiler doesn't see, and are read back as ordinary memory: a wait for requests lies between in the listing."""
    if not os.path.exists(build.LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    kernel, seen = "lin_tile_kernelILi2E", 0
    for code in code_objects(build.LIB):
        if kernel.encode() not in code:
            continue
        (tmp_path / "code.o").write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", str(tmp_path / "code.o")], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
            if kernel in part.split("\n", 1)[0]:
                behind = re.split(r"\sglobal_load_lds_dword\s", part)[1:]
                assert len(behind) >= 2 and all("vmcnt(" in b.split("ds_read_b32")[0] for b in behind), part.split("\n", 1)[0]
                seen += 1
    assert seen, f"{kernel}: not in {build.LIB}"
