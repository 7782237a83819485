"""What the compiler reports about the built kernels: a prompt kernel whose operands land in scratch waits for memory inside its main loop."""
import os
import re
import struct
import subprocess

import pytest

from ktransformers_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def private_segments(lib, tmp):
    """{mangled kernel name: bytes of scratch per lane} over the gfx950 code objects of a library."""
    data = open(lib, "rb").read()
    out = {}
    for m in re.finditer(MAGIC, data):
        at = m.start()
        pos, (n,) = at + 32, struct.unpack_from("<Q", data, at + 24)
        for _ in range(n):
            ofs, size, idlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if size and b"gfx950" in triple:
                tmp.write_bytes(data[at + ofs:at + ofs + size])
                notes = subprocess.run([READELF, "--notes", str(tmp)], check=True, capture_output=True, text=True).stdout
                for k in re.split(r"\n\s+- \.", notes):
                    name, priv = re.search(r"\.?name:\s+(_Z\S+)", k), re.search(r"private_segment_fixed_size:\s+(\d+)", k)
                    if name and priv:
                        out[name.group(1)] = int(priv.group(1))
    return out


@pytest.mark.parametrize("kernel", ["moe_gguf_fold_kernel", "moe_rawint4_chunk_kernel", "mla_decode_wide_kernel", "lin_tile_kernel", "moe_gemm_stream_kernel", "moe_fp8_stream_kernel", "mla_prefill_kernelILb1E"])
def test_prompt_kernels_keep_their_operands_in_registers(kernel, tmp_path):
    if not os.path.exists(build.LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    seen = {k: v for k, v in private_segments(build.LIB, tmp_path / "code.o").items() if kernel in k}
    assert seen, f"{kernel}: not in {build.LIB}"
    assert not {k: v for k, v in seen.items() if v}, "scratch bytes per lane"
