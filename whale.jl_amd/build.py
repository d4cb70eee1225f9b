"""Builds the package's native libraries in-tree.

    libwhale_amd.so    C ABI + gfx950 kernels (hipcc --offload-arch=gfx950)
    libwhale_synth.so  seeded synthetic workload generator (host only, g++)

Run as `python whale.jl_amd/build.py` or through __graft_entry__.build().
"""
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed FP32 VALU ops stay off in every HIP build of this project
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]
# The DP kernels are at the register limit of their occupancy, so the order of
# their instructions and what is hoisted decide how long a row takes.  Measured
# against -O3 and the default schedule for all, per pass: FP64, one family of
# 240 genes 1436 -> 1365 us, 12 families 401 -> 385, 1000 families
# log-likelihood 447 -> 420; FP32, 5000 families 2955 -> 2893, 10,000 families
# 8750 -> 8630; scaled FP64, 777 families 1580 -> 1563.  (FP32 with the
# schedule of FP64 is 5 % slower, with -O1 1 % slower.)
_ILP = ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"]
SOURCE_FLAGS = {"dp_fp64.hip": ["-O1"] + _ILP, "dp_fp32.hip": ["-O2"], "dp_fp64s.hip": _ILP}
MAIN_SOURCES = ("dp_fp64.hip", "dp_fp32.hip", "dp_fp64s.hip", "kernels.hip", "capi.cpp", "host.cpp")


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def build_main(out=None):
    """One object per source, compiled side by side, then the library."""
    out = out or os.path.join(HERE, "libwhale_amd.so")
    tmp = out + ".tmp"
    with tempfile.TemporaryDirectory() as d:
        objs = [os.path.join(d, f + ".o") for f in MAIN_SOURCES]
        with ThreadPoolExecutor(len(objs)) as ex:
            list(ex.map(lambda so: _run([HIPCC] + HIP_FLAGS + SOURCE_FLAGS.get(so[0], []) +
                                        ["-c", os.path.join(CSRC, so[0]), "-o", so[1]]), zip(MAIN_SOURCES, objs)))
        _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", tmp, "-lpthread"])
    os.replace(tmp, out)
    return out


def build_synth(out=None):
    out = out or os.path.join(HERE, "libwhale_synth.so")
    tmp = out + ".tmp"
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", os.path.join(CSRC, "synth.cpp"), "-o", tmp,
          "-lpthread"])
    os.replace(tmp, out)
    return out


def build_all():
    return build_main(), build_synth()


if __name__ == "__main__":
    what = sys.argv[1:] or ["all"]
    if "all" in what or "main" in what:
        build_main()
    if "all" in what or "synth" in what:
        build_synth()
