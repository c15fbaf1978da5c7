"""Build the HIP engine library (``libmba.so``) in-tree for gfx950."""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmba.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-std=c++17", "-O3", "--offload-arch=gfx950", "-fPIC",
    # Packed FP32 instructions stay off on this target.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
SOURCES = ["mba_engine.hip", "mba_prep.hip", "mba_io.cpp"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed building libmba.so")


def build(verbose: bool = False) -> str:
    """Compile the sources side by side and link them."""
    with tempfile.TemporaryDirectory() as tmp:
        objs = [os.path.join(tmp, s + ".o") for s in SOURCES]
        with concurrent.futures.ThreadPoolExecutor(len(SOURCES)) as pool:
            list(pool.map(lambda so: _run([HIPCC, *FLAGS, "-c", "-o", so[1], os.path.join(CSRC, so[0])], verbose),
                          zip(SOURCES, objs)))
        lib = LIB + ".tmp"
        _run([HIPCC, "--offload-arch=gfx950", "-fPIC", "-shared", "-o", lib, *objs], verbose)
    os.replace(lib, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
