"""Build libsamfast.so (HIP kernels + C ABI) and the host module _samfast_host.so in-tree for gfx950.

Usage: python segment-anything-fast_amd/build.py [--force]
hipcc cross-compiles without a GPU; the shared objects land next to the Python
package (samfast_amd/lib/) so that they travel with the tree.
"""

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
INCLUDE = HERE.parent / "include"
LIB_DIR = HERE / "samfast_amd" / "lib"
LIB_PATH = LIB_DIR / "libsamfast.so"
HOST_SRC = CSRC / "host_torch.cpp"
HOST_PATH = LIB_DIR / "_samfast_host.so"
OBJ_DIR = HERE / "build"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    f"-I{INCLUDE}", f"-I{CSRC}",
]


def sources():
    return sorted(CSRC.glob("*.hip"))


def _compile(src: Path) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [HIPCC, *FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_host() -> Path:
    """The CPython module over torch's C++ API (host code only, no device code in it)."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    lib_dir = Path(torch.__file__).resolve().parent / "lib"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{INCLUDE}",
           f"-I{sysconfig.get_paths()['include']}", *(f"-isystem{p}" for p in cpp_extension.include_paths()),
           "-isystem/opt/rocm/include", str(HOST_SRC), "-o", str(HOST_PATH), f"-L{lib_dir}",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on {HOST_SRC.name}:\n{res.stderr}")
    if res.stderr.strip():
        sys.stderr.write(res.stderr + "\n")
    return HOST_PATH


def build(force: bool = True, jobs: int = 4) -> Path:
    """Compile every .hip under csrc/, link libsamfast.so and build the host module.  Returns the
    library's path."""
    srcs = sources()
    deps = srcs + [HOST_SRC] + list(CSRC.glob("*.hpp")) + list(INCLUDE.glob("*.h"))
    if not force and LIB_PATH.exists() and HOST_PATH.exists():
        newest = max(p.stat().st_mtime for p in deps)
        if min(LIB_PATH.stat().st_mtime, HOST_PATH.stat().st_mtime) >= newest:
            return LIB_PATH
    OBJ_DIR.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host)
        objs = list(pool.map(_compile, srcs))
        host.result()
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(LIB_PATH)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    return LIB_PATH


if __name__ == "__main__":
    path = build(force="--force" in sys.argv or True)
    print(path)
