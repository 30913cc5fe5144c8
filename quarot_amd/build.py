"""Build recipe: libquarot_hip.so by plain hipcc, gfx950 only, no torch headers; and _host.so, the CPython module of the
hot entry points' host side (csrc/host.cpp), by g++ against torch's headers.

    python -m quarot_amd.build                # compile every source, link in-tree (quarot_amd/libquarot_hip.so)
    python -m quarot_amd.build --incremental  # recompile only sources newer than their objects
"""
import concurrent.futures
import os
import pathlib
import subprocess
import sys

PKG = pathlib.Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB = PKG / "libquarot_hip.so"
HOST = PKG / "_host.so"
OBJ = PKG.parent / "build" / "obj"
SOURCES = ("api.hip", "quant.hip", "gemm.hip", "gemm_mid.hip", "gemm_e2m3.hip", "gemm_x6.hip", "gemm_f6.hip", "hadamard.hip", "kv.hip", "attn.hip", "calib.hip", "decode_fused.hip",
           "paged_f16.hip")
FLAGS = ("--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-fno-gpu-rdc",
         # every fp16/fp32 operation must round on its own (the reference's results are defined that
         # way): no fused multiply-add contraction unless a kernel spells fma out
         "-ffp-contract=off",
         # a kernel's leading arguments arrive in scalar registers with its waves (up to 16 dwords, structures excepted) instead of
         # by a load that everything waits for: 333 x 4096 x 4096 x 3 behind two fronts 36.3 -> 35.0 us, 48 x 13824 x 5120 20.3 -> 19.7
         "-mllvm", "-amdgpu-kernarg-preload-count=16",
         # packed-fp32 VALU forms are kept out of the generated code on purpose
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument")


def _host_commands():
    """(compile, link) of _host.so: one object, then the link against libquarot_hip.so beside it."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    src, obj = CSRC / "host.cpp", OBJ / "host.o"
    include = [f"-I{d}" for d in (*cpp_extension.include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"])]
    compile_ = ["g++", "-O2", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *include, "-c", str(src), "-o", str(obj)]
    torch_lib = pathlib.Path(torch.__file__).resolve().parent / "lib"
    link = ["g++", "-shared", str(obj), "-o", str(HOST), f"-L{torch_lib}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip",
            f"-L{PKG}", f"-l:{LIB.name}", "-Wl,-rpath,$ORIGIN"]
    return src, obj, compile_, link


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature: harmless, filtered.
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({res.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def build(verbose=True, incremental=False):
    """One object per source (compiled side by side), then one link.  incremental: a source is
    recompiled only if it, or any header beside it, is newer than its object."""
    OBJ.mkdir(parents=True, exist_ok=True)
    headers_mtime = max((h.stat().st_mtime for h in CSRC.glob("*.h")), default=0.0)
    jobs, objs = [], []
    for s in SOURCES:
        src, obj = CSRC / s, OBJ / (s[:-4] + ".o")
        objs.append(str(obj))
        fresh = incremental and obj.exists() and obj.stat().st_mtime > max(src.stat().st_mtime, headers_mtime)
        if not fresh:
            jobs.append(["hipcc", *FLAGS, "-c", str(src), "-o", str(obj)])
    host_src, host_obj, host_compile, host_link = _host_commands()
    header = PKG.parent / "include" / "quarot_hip.h"
    if not (incremental and host_obj.exists() and host_obj.stat().st_mtime > max(host_src.stat().st_mtime, header.stat().st_mtime)):
        jobs.append(host_compile)
    workers = max(1, min(len(jobs), (os.cpu_count() or 2)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=workers) as pool:
        list(pool.map(lambda c: _run(c, verbose), jobs))
    _run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *objs, "-o", str(LIB)], verbose)
    _run(host_link, verbose)
    return LIB


if __name__ == "__main__":
    build(incremental="--incremental" in sys.argv)
