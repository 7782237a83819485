"""Build the gfx950 shared library (hipcc cross-compiles without a GPU).

    python -m ktransformers_amd.build [--force]

Every csrc/*.hip is compiled to its own object (in parallel, only when it or a header it may include changed) and the
objects are linked into ktransformers_amd/lib/libktx_hip.so (git-ignored).
"""
from __future__ import annotations

import glob
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(LIBDIR, "obj")
LIB = os.path.join(LIBDIR, "libktx_hip.so")
# the sequence-mixer, hybrid-decoder, window-attention / scan and decayed-state kernels alone (include/ktx_seq.h, ktx_hyb.h, ktx_swa.h,
# ktx_gla.h): what the fp32-residual families need, built in about a minute
SEQ_LIB = os.path.join(LIBDIR, "libktx_seq.so")
HOST_SOURCE = os.path.join(CSRC, "ktx_host.cpp")
SEQ_SOURCES = ("ktx_seq.hip", "ktx_hyb.hip", "ktx_swa.hip", "ktx_gla.hip", "ktx_err.hip")

# -ffp-contract=off: the parity contract needs every fp32 op rounded exactly as the reference's AVX512 code does;
# FMAs appear only where the reference issues one (explicit fmaf()).
# No packed fp32 instructions: some forms of v_pk_{add,mul,fma}_f32, which -O3 makes from ordinary float code, have given wrong results
# on this hardware now and then (hipcc's host pass warns that it does not know the feature: harmless).
CFLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-fPIC", "-Wno-unused-value",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def _headers() -> list[str]:
    return (glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.inc"))
            + glob.glob(os.path.join(HERE, "..", "include", "*.h")))


def _deps(src: str, seen: set | None = None) -> list[str]:
    """The headers a source reaches through its quoted #include lines (searched beside the including file and in include/)."""
    import re
    seen = set() if seen is None else seen
    out = []
    try:
        text = open(src, encoding="utf-8", errors="replace").read()
    except OSError:
        return out
    for inc in re.findall(r'^\s*#\s*include\s*"([^"]+)"', text, flags=re.M):
        for base in (os.path.dirname(src), CSRC, os.path.join(HERE, "..", "include")):
            path = os.path.normpath(os.path.join(base, inc))
            if os.path.exists(path):
                if path not in seen:
                    seen.add(path)
                    out.append(path)
                    out.extend(_deps(path, seen))
                break
    return out


def _obj(src: str) -> str:
    return os.path.join(OBJDIR, os.path.basename(src)[:-4] + ".o")


def _stale(target: str, deps: list[str]) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def build_seq(force: bool = False, verbose: bool = False) -> str:
    """libktx_seq.so from SEQ_SOURCES only (ktransformers_amd._native_seq loads it when libktx_hip.so is absent)."""
    srcs = [os.path.join(CSRC, n) for n in SEQ_SOURCES]
    if not force and not _stale(SEQ_LIB, [d for s in srcs for d in [s] + _deps(s)]):
        return SEQ_LIB
    os.makedirs(OBJDIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

    def compile_one(src: str) -> None:
        cmd = [hipcc, *CFLAGS, "-c", src, "-o", _obj(src)]
        if verbose:
            print(" ".join(cmd), file=sys.stderr)
        subprocess.run(cmd, check=True)

    todo = [s for s in srcs if force or _stale(_obj(s), [s] + _deps(s))]
    with ThreadPoolExecutor(max_workers=max(1, min(len(todo), os.cpu_count() or 4))) as ex:
        list(ex.map(compile_one, todo))
    tmp = SEQ_LIB + f".tmp{os.getpid()}"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *[_obj(s) for s in srcs], "-o", tmp], check=True)
    os.replace(tmp, SEQ_LIB)
    return SEQ_LIB


def host_lib() -> str:
    """Where the host module of this interpreter and this torch lies: it has both's layouts compiled in, so that another one's is not found."""
    import sysconfig

    import torch
    return os.path.join(LIBDIR, f"ktx_host-{torch.__version__}{sysconfig.get_config_var('EXT_SUFFIX')}")


def build_host(force: bool = False, verbose: bool = False) -> str:
    """The CPython module of the host side (csrc/ktx_host.cpp, against this interpreter's and torch's headers)."""
    target = host_lib()
    if not force and not _stale(target, [HOST_SOURCE, __file__] + _deps(HOST_SOURCE)):
        return target
    import sysconfig

    from torch.utils.cpp_extension import include_paths, library_paths
    os.makedirs(LIBDIR, exist_ok=True)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    tmp = target + f".tmp{os.getpid()}"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           *[f"-I{d}" for d in include_paths() + [os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]], HOST_SOURCE, "-o", tmp,
           *[f"-L{d}" for d in library_paths()], "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), file=sys.stderr)
    subprocess.run(cmd, check=True)
    os.replace(tmp, target)
    return target


def needs_build() -> bool:
    return _stale(LIB, sources() + _headers())


def build(force: bool = False, verbose: bool = False) -> str:
    """libktx_hip.so, and the host module beside it where there are a compiler and headers for it: without it every call is made from Python."""
    lib = _build_lib(force, verbose)
    try:
        build_host(force, verbose)
    except (OSError, ImportError, subprocess.CalledProcessError) as e:
        print(f"ktransformers_amd: {os.path.basename(HOST_SOURCE)} was not built ({e}); short calls take the host longer without it", file=sys.stderr)
    return lib


def _build_lib(force: bool, verbose: bool) -> str:
    if not force and not needs_build():
        return LIB
    os.makedirs(OBJDIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    hdrs = _headers()
    todo = [s for s in sources() if force or _stale(_obj(s), [s] + (_deps(s) or hdrs))]

    def compile_one(src: str) -> None:
        cmd = [hipcc, *CFLAGS, "-c", src, "-o", _obj(src)]
        if verbose:
            print(" ".join(cmd), file=sys.stderr)
        subprocess.run(cmd, check=True)

    with ThreadPoolExecutor(max_workers=max(1, min(len(todo), os.cpu_count() or 4))) as ex:
        list(ex.map(compile_one, todo))
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *[_obj(s) for s in sources()], "-o", LIB]
    if verbose:
        print(" ".join(cmd), file=sys.stderr)
    subprocess.run(cmd, check=True)
    return LIB


if __name__ == "__main__":
    if "--seq" in sys.argv:
        print(build_seq(force="--force" in sys.argv, verbose=True))
    else:
        print(build(force="--force" in sys.argv, verbose=True))
