"""Build the in-tree HIP library libkvq_int8.so for gfx950 (hipcc, no JIT cache) and the CPython module
_torch_calls.so that calls it with torch tensors (host code).

Run as a script (python int8-kvcache_amd/build.py) or through __graft_entry__.build(). Both land next to
this file's kvq/ package so that they travel with the source tree.
"""
import importlib.util
import os
import re
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "kvq_int8.hip")
OUT = os.path.join(HERE, "kvq", "libkvq_int8.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-ffp-contract=off",                               # every fma in the kernels is written out
    "-fhip-fp32-correctly-rounded-divide-sqrt",        # x / s is IEEE division (bit-exact codes)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",             # MFMA results in VGPRs (no v_accvgpr_read copies)
]


CALLS_SRC = os.path.join(HERE, "csrc", "torch_calls.cpp")
CALLS_OUT = os.path.join(HERE, "kvq", "_torch_calls.so")
CXX = os.environ.get("KVQ_CXX", "/opt/rocm/bin/amdclang++")


def _calls_flags():
    torch_dir = os.path.dirname(importlib.util.find_spec("torch").origin)
    with open(os.path.join(torch_dir, "version.py")) as f:   # torch.__version__ without importing torch
        version = re.search(r"^__version__ = ['\"](.+)['\"]", f.read(), re.M).group(1)
    return ["-O2", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f'-DKVQ_TORCH_VERSION="{version}"', f"-I{torch_dir}/include", "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}",
            f"-L{torch_dir}/lib", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def build(verbose=False):
    """Compile both. An output whose compilation failed is removed: a file of an earlier build beside a new one
    would be called with signatures that are no longer the library's."""
    jobs = []
    for cmd, out in (([HIPCC, *FLAGS, SRC], OUT), ([CXX, CALLS_SRC, *_calls_flags()], CALLS_OUT)):
        cmd = [*cmd, "-o", out + ".tmp"]
        if verbose:
            print(" ".join(cmd), flush=True)
        jobs.append((subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True), out))
    failed = []
    for job, out in jobs:
        text = job.communicate()[0]
        if job.returncode != 0:
            failed.append(f"building {os.path.basename(out)} failed ({job.returncode}):\n{text[-4000:]}")
            for path in (out, out + ".tmp"):
                if os.path.exists(path):
                    os.remove(path)
        else:
            os.replace(out + ".tmp", out)
    if failed:
        raise RuntimeError("\n".join(failed))
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
