"""Builds the HIP library (csrc/*.hip -> csrc/libqwen_tailor_hip.so) for gfx950 with hipcc and the host module (csrc/host.cpp ->
csrc/_qt_host.so) with g++, in-tree."""
from __future__ import annotations

import glob
import hashlib
import os
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
SO = os.path.join(CSRC, "libqwen_tailor_hip.so")
HOST_SO = os.path.join(CSRC, "_qt_host.so")
HEADER = os.path.join(os.path.dirname(os.path.dirname(CSRC)), "include", "qwen_tailor_hip.h")
# kernel arguments come in scalar registers with the launch instead of by a load at the head of every wavefront: 5 x 3 step 243.5 -> 236.5 us, 16 x 4
# 416.0 -> 409.4, prefill of 61 tokens 19.75 -> 19.2, of 2048 49.8 -> 49.0
FLAGS = ["-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-mllvm", "-amdgpu-kernarg-preload-count=16", "-Wno-unused-command-line-argument"]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]


HASH = SO + ".srchash"


def host_abi() -> str:
    """what the host module is compiled against besides its source: torch's version and its C++ ABI, HIP's version, CPython's ABI"""
    import torch
    return " ".join(map(str, (torch.__version__, torch.version.hip, torch._C._GLIBCXX_USE_CXX11_ABI, sysconfig.get_config_var("SOABI"))))


def source_hash() -> str:
    """sha256 over the names and contents of every source the libraries are built from (csrc/*.hip, *.h, *.cpp and the C header), the
    flags and what the host module is compiled against"""
    h = hashlib.sha256(" ".join([*FLAGS, *HOST_FLAGS, host_abi()]).encode())
    for path in sorted(p for kind in ("*.hip", "*.h", "*.cpp") for p in glob.glob(os.path.join(CSRC, kind))) + [HEADER]:
        h.update(os.path.basename(path).encode())
        with open(path, "rb") as f:
            h.update(f.read())
    return h.hexdigest()


def is_current() -> bool:
    """True if the built libraries exist and were built from the sources, and for the torch and the Python, as they are now."""
    try:
        with open(HASH) as f:
            return os.path.exists(SO) and os.path.exists(HOST_SO) and f.read().strip() == source_hash()
    except OSError:
        return False


def _hipcc():
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.sep not in c or os.path.exists(c)):
            return c
    raise RuntimeError("hipcc not found")


def build(verbose: bool = False, jobs: int = 8) -> str:
    """Compile every csrc/*.hip and link them into one shared library, and the host module against it.  Always recompiles."""
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    hipcc = _hipcc()
    digest = source_hash()                  # taken before compiling: an edit made during the build leaves the library stale
    objs = [s[:-4] + ".o" for s in srcs]

    def one(pair):
        src, obj = pair
        cmd = [hipcc, *FLAGS, "-c", src, "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
        if verbose and r.stderr.strip():
            print(r.stderr)

    with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(srcs)))) as ex:
        list(ex.map(one, zip(srcs, objs)))
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", SO + ".tmp"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(SO + ".tmp", SO)
    _build_host()
    with open(HASH, "w") as f:
        f.write(digest + "\n")
    return SO


def _build_host():
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [sysconfig.get_paths()["include"], os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           "/opt/rocm/include"]
    cmd = [os.environ.get("CXX", "g++"), *HOST_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{p}" for p in inc),
           os.path.join(CSRC, "host.cpp"), "-o", HOST_SO + ".tmp", f"-L{os.path.join(root, 'lib')}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip",
           "-ltorch_python", f"-L{CSRC}", "-lqwen_tailor_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for host.cpp:\n{r.stdout}\n{r.stderr}")
    os.replace(HOST_SO + ".tmp", HOST_SO)


if __name__ == "__main__":
    print(build(verbose=True))
