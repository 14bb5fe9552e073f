"""Build liblandmark_hip.so for gfx950 with plain hipcc (cross-compiles without a GPU) and _native.so, the host
path of the Python shim, with g++ against torch's headers.

    python landmark-attention_amd/build.py [--force]

One object per HIP translation unit in csrc/, linked into
landmark_hip/liblandmark_hip.so next to the Python shim that loads it; _native.so sits beside it and calls it.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "landmark_hip", "liblandmark_hip.so")
NATIVE_SRC = os.path.join(CSRC, "lmk_torch.cpp")
NATIVE_OUT = os.path.join(HERE, "landmark_hip", "_native.so")
OBJ = os.path.join(HERE, "build")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-math-errno", "-ffp-contract=fast",
    # packed fp32 VALU ops are switched off for every device compile of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-attributes", "-Wno-ignored-optimization-argument",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err:
        print(err, file=sys.stderr)
    return obj


def _compile_native() -> str:
    import sysconfig

    from torch.utils import cpp_extension
    import torch
    obj = os.path.join(OBJ, "lmk_torch.o")
    includes = [f"-I{d}" for d in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include")]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, "-c", NATIVE_SRC, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed for lmk_torch.cpp:\n" + r.stderr)
    return obj


def _link_native(obj: str) -> None:
    from torch.utils import cpp_extension
    libs = cpp_extension.library_paths()
    cmd = ["g++", "-shared", "-o", NATIVE_OUT, obj, *(f"-L{d}" for d in libs), "-ltorch_python", "-ltorch", "-ltorch_cpu",
           "-ltorch_hip", "-lc10", "-lc10_hip", f"-L{os.path.dirname(OUT)}", "-l:liblandmark_hip.so", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link of _native.so failed:\n" + r.stderr)


def build(force: bool = True, jobs: int = 4) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    if not force and os.path.exists(OUT) and os.path.exists(NATIVE_OUT):
        newest = max(os.path.getmtime(os.path.join(CSRC, f)) for f in os.listdir(CSRC))
        if min(os.path.getmtime(OUT), os.path.getmtime(NATIVE_OUT)) >= newest:
            return OUT
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(_compile_native)
        objs = list(ex.map(_compile, srcs))
        native_obj = native.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", OUT, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    _link_native(native_obj)
    return OUT


if __name__ == "__main__":
    print(build(force="--force" in sys.argv or True))
