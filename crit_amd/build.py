"""Builds libcrit_pkv.so (the C-ABI library of gfx950 kernels) with hipcc, in-tree, one object per source in parallel.

    python -m crit_amd.build            # compile everything, link crit_amd/lib/libcrit_pkv.so

With it goes _pkv_host.so, the native share of the package's host code, which takes g++ and the headers of Python and torch
and is optional: where it does not compile the build says so and the package's Python code does it all. With $CRIT_PKV_OUT the
library alone is linked, there, and the two in crit_amd/lib stay as they are.

hipcc cross-compiles for gfx950 without a GPU. No fast-math; FP contraction is off so that every fused multiply-add in
the kernels is one the source spells out (a column's bits must not depend on which template instance computed it).
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "libcrit_pkv.so")
OBJ_DIR = os.path.join(LIB_DIR, "obj")

# (--offload-compress: the device code is stored compressed and unpacked by the HIP runtime when a source file's kernels
# are first used: the library is 8 MB instead of 26)
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "--offload-compress",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"]

# The window and prompt kernels' accumulators are rescaled by the vector pipe between products, which cannot reach the
# registers that the compiler keeps products in for kernels of one wavefront a SIMD (160 moves a pair of steps with three
# query tiles; prompt chunks of 256-wide heads 104 bytes of scratch a lane, and 97.4 -> 91.3 us without, 254 -> 222 over
# fp8:row pages): their products take ordinary registers. The bits are the same. (An internal option of this image's
# compiler: one that does not know it stops with "Unknown command line argument", and is to be run without.)
OWN_FLAGS = {start: ["-mllvm", "-amdgpu-mfma-vgpr-form=1"] for start in ("pkv_attend_", "pkv_prefill")}


HOST_LIB = os.path.join(LIB_DIR, "_pkv_host.so")


def _compile_host():
    """The native share of the package's host code: a Python extension module against this interpreter and this torch. The old
    one goes first (a module that does not match the library is worse than none); the new one is there whole or not at all."""
    if os.path.exists(HOST_LIB):
        os.remove(HOST_LIB)
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    part = f"{HOST_LIB}.{os.getpid()}"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f'-DCRIT_TORCH_VERSION="{torch.__version__}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + sysconfig.get_paths()["include"],
           *["-isystem" + path for path in include_paths()], os.path.join(CSRC, "pkv_host.cpp"), "-o", part,
           *["-L" + path for path in library_paths()], "-ltorch_python", "-ltorch_cpu", "-lc10"]
    done = subprocess.run(cmd, capture_output=True, text=True)
    if done.returncode:
        raise RuntimeError(f"g++ failed on pkv_host.cpp:\n{done.stderr}")
    os.replace(part, HOST_LIB)


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src):
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    own = [f for start, flags in OWN_FLAGS.items() if os.path.basename(src).startswith(start) for f in flags]
    cmd = ["hipcc", *FLAGS, *own, *os.environ.get("CRIT_PKV_EXTRA_FLAGS", "").split(), "-c", src, "-o", obj]
    done = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in done.stderr.splitlines() if noise not in line)
    if done.returncode:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    return obj, err


def build(verbose=True, jobs=None):
    """Compile every .hip under csrc/ for gfx950 and link the shared library; returns its path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    out = os.environ.get("CRIT_PKV_OUT", LIB)
    jobs = jobs or min(8, os.cpu_count() or 1)
    with ThreadPoolExecutor(jobs) as pool:
        host = pool.submit(_compile_host) if os.path.abspath(out) == LIB else None
        found = list(pool.map(_compile, sources()))
    for _, err in found:
        if err.strip() and verbose:
            print(err, file=sys.stderr)
    link = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *[obj for obj, _ in found]]
    done = subprocess.run(link, capture_output=True, text=True)
    if done.returncode:
        raise RuntimeError(f"link failed:\n{done.stderr}")
    if host is not None and host.exception() is not None:
        print(f"without the native host code, which is optional: {host.exception()}", file=sys.stderr)
    if verbose:
        print(f"built {out}")
    return out


if __name__ == "__main__":
    build()
