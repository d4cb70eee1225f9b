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
            list(ex.map(lambda so: _run([HIPCC] + HIP_FLAGS + ["-c", os.path.join(CSRC, so[0]), "-o", so[1]]),
                        zip(MAIN_SOURCES, objs)))
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
