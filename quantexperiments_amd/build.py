"""Ahead-of-time build of libsqhip.so for gfx950 (hipcc) and of the torch extension over it (g++); no JIT."""

from __future__ import annotations

import os
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "libsqhip.so"
NATIVE = HERE / "_native.so"
SOURCES = ["sq_api.hip", "sq_dequant.hip", "sq_planes.hip", "sq_plane_product.hip", "sq_small_generic.hip", "sq_gemv.hip", "sq_gemv_b16d8.hip",
           "sq_gemv_b12d4.hip", "sq_gemv_b10d4.hip", "sq_gemv_b8d4.hip", "sq_gemm.hip", "sq_gemm256.hip", "sq_stream.hip", "sq_stream_build.hip", "sq_relabel.hip",
           "sq_q8.hip", "sq_neighbours.hip", "sq_segs.hip", "sq_sieve.hip", "sq_mid.hip", "sq_mid_b16d8.hip", "sq_mid_b12d4.hip", "sq_mid_b10d4.hip", "sq_mid_b8d4.hip",
           "sq_mid_dense.hip", "sq_fused.hip", "sq_fused_b16d8.hip", "sq_fused_b12d4.hip", "sq_fused_b10d4.hip", "sq_fused_b8d4.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.sep not in c or os.path.exists(c)):
            return c
    raise RuntimeError("hipcc not found")


def _native_command() -> list:
    """g++ line of the torch extension (host code only: it calls libsqhip.so, which it finds next to itself)."""
    import sysconfig
    import torch
    t = Path(torch.__file__).parent
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{t}/include", f"-I{t}/include/torch/csrc/api/include",
            f"-I{sysconfig.get_paths()['include']}", f"-isystem{rocm}/include", str(CSRC / "sq_torch.cpp"), "-o", str(NATIVE), f"-L{t}/lib", "-lc10",
            "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python", f"-L{HERE}", "-lsqhip", "-Wl,-rpath,$ORIGIN", f"-L{rocm}/lib",
            "-lamdhip64"]


def build(verbose: bool = False, extra_flags: tuple = ()) -> Path:
    """Compile every kernel translation unit, link libsqhip.so next to this file and build _native.so beside it."""
    hipcc = _hipcc()
    objdir = CSRC / "build"
    objdir.mkdir(exist_ok=True)

    def one(src: str) -> Path:
        obj = objdir / (Path(src).stem + ".o")
        cmd = [hipcc, *FLAGS, *extra_flags, "-c", str(CSRC / src), "-o", str(obj)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{err}")
        if verbose and err.strip():
            print(err)
        return obj

    with ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 4)) as ex:
        objs = list(ex.map(one, SOURCES))
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB), *map(str, objs)],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    r = subprocess.run(_native_command(), capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on sq_torch.cpp:\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
