"""Build libldo_hip.so for gfx950 in-tree (latticednaorigami_amd/lib/)."""
import os
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "libldo_hip.so")
SOURCES = ["sweep_all.hip", "sweep_std.hip", "sampler.hip", "mlp.hip", "plan.cpp", "tables.cpp"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # identical FP64 arithmetic to the reference's x86 build: no FMA fusion
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


DRIVER = os.path.join(LIB_DIR, "ldo_run")


def build(verbose=False):
    os.makedirs(LIB_DIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    tmp = LIB + ".tmp"

    def run(cmd):
        if verbose:
            print(" ".join(cmd))
        subprocess.run(cmd, check=True)

    with tempfile.TemporaryDirectory() as d, ThreadPoolExecutor(len(SOURCES)) as pool:
        objs = [os.path.join(d, s + ".o") for s in SOURCES]
        jobs = [pool.submit(run, [hipcc, *HIPCC_FLAGS, "-x", "hip", "-c", "-o", o,
                                  os.path.join(CSRC, s)]) for s, o in zip(SOURCES, objs)]
        for j in jobs:
            j.result()
        run([hipcc, "--offload-arch=gfx950", "-shared", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    # the reference-compatible driver: host C++ over the C ABI
    cmd = ["g++", "-O2", "-std=c++17", "-o", DRIVER + ".tmp",
           os.path.join(CSRC, "driver", "ldo_run.cpp"), "-L" + LIB_DIR, "-lldo_hip",
           "-Wl,-rpath,$ORIGIN"]
    run(cmd)
    os.replace(DRIVER + ".tmp", DRIVER)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
