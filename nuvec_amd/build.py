"""Compiles the gfx950 kernels and the C ABI into `nuvec_amd/libnuvec_hip.so` with hipcc, and the Python package's native
calls (`csrc/native.cpp`, torch's C++ interface over that C ABI) into `nuvec_amd/_native.so` with the host compiler.

Cross-compiles without a GPU.  Run as `python -m nuvec_amd.build` or through
`__graft_entry__.build()`.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(HERE, "..", "include")
LIB = os.path.join(HERE, "libnuvec_hip.so")
NATIVE = os.path.join(HERE, "_native.so")
SOURCES = ["qmg_b8.hip", "qmg_b6.hip", "qmg_b5.hip", "qmg_b4.hip", "qmg_b3.hip", "qmg_b2.hip", "qmg_b1.hip", "qmg_nvfp4.hip", "qmg_fp8.hip", "qmg_fp4.hip",
           "qms_b8.hip", "qms_b6.hip", "qms_b5.hip", "qms_b4.hip", "qms_b3.hip", "qms_b2.hip", "qms_fp4.hip", "qms_fp8.hip", "qms_nvfp4.hip", "qms.hip",
           "qmf_b8.hip", "qmf_fp8.hip", "qmf_b6.hip", "qmf_b5.hip", "qmf_b4.hip", "qmf_fp4.hip", "qmf_nvfp4.hip", "qmf_b3.hip", "qmf_b2.hip", "qmf_b1.hip", "qmm.hip", "qmv.hip", "qmv_dot8.hip", "qmm_f32.hip", "qmm_dense.hip", "qmr.hip",
           "qvm.hip", "nvq_api.hip", "affine_quant.hip", "fp_quant.hip", "qmf.hip", "gather.hip", "repack.hip", "calib.hip", "qattn.hip", "qattn_prompt.hip", "qattn_prompt_f32.hip", "qmd.hip", "glu.hip"]  # slowest to compile first

# -ffp-contract=off: the quantizers must round every operation as the CPU does; fused
# multiply-adds are written explicitly where wanted.  Correctly rounded f32 division is
# hipcc's default and is spelled out because the bit-exact quantizers depend on it.
# Packed-FP32 instructions are switched off for all device code.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt", "-fno-gpu-flush-denormals-to-zero",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-inline-asm", "-fvisibility=hidden",
    f"-I{INCLUDE}", f"-I{CSRC}",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _link(cmd, target: str, what: str) -> None:
    """Runs `cmd`, which ends in `-o`, into a name of this process beside `target` and puts the whole file there: processes that find
    the library missing and build it together load either a complete one or none."""
    part = f"{target}.{os.getpid()}"
    try:
        proc = subprocess.run([*cmd, part], capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"{what}:\n{proc.stdout}\n{proc.stderr}")
        os.replace(part, target)
    finally:
        if os.path.exists(part):
            os.remove(part)


def build(verbose: bool = False, jobs: int = 8, changed_only: bool = False) -> str:
    """Compiles every source and links the library.  `changed_only` (a development aid, `--changed` on the command line):
    sources older than their object files are not compiled again, unless a header is newer than the object."""
    hipcc = _hipcc()
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    headers = [os.path.join(d, f) for d in (CSRC, INCLUDE) for f in os.listdir(d) if f.endswith(".h")]
    newest_header = max(os.path.getmtime(h) for h in headers)

    def compile_one(src):
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        if changed_only and os.path.exists(obj) and os.path.getmtime(obj) > max(newest_header, os.path.getmtime(os.path.join(CSRC, src))):
            return obj
        cmd = [hipcc, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{proc.stdout}\n{proc.stderr}")
        # hipcc's host pass warns that it does not know the packed-fp32 feature: harmless.
        noise = "is not a recognized feature for this target"
        err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l and l.strip())
        if verbose and err:
            print(err, file=sys.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(compile_one, SOURCES))
    _link([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o"], LIB, "link failed")
    build_native(verbose)
    return LIB


def build_native(verbose: bool = False) -> str:
    """Compiles `csrc/native.cpp` against the installed torch; links to the library beside it."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-I{root}/include", "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}", f"-I{INCLUDE}",
           os.path.join(CSRC, "native.cpp"), f"-L{root}/lib", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip",
           "-ltorch_python", f"-L{HERE}", "-l:libnuvec_hip.so", "-Wl,-rpath,$ORIGIN", "-o"]
    if verbose:
        print(" ".join([*cmd, NATIVE]), flush=True)
    _link(cmd, NATIVE, "g++ failed on native.cpp")
    return NATIVE


if __name__ == "__main__":
    print(build(verbose=True, changed_only="--changed" in sys.argv))
