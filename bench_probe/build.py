"""Build bench_probe/librtb_probe.so, the benchmark's measurement aid (not part
of the library): the attainable matrix-core rates of the device
(independent MFMA chains) and the host's page-cache read ceiling for a file.
bench.py loads it; the product never does."""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "librtb_probe.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build(verbose: bool = False) -> str:
    tmp = LIB + ".tmp"
    subprocess.run([HIPCC, "-O3", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    # accumulators stay in VGPRs: without it each MFMA of a chain pays
                    # copies to and from AGPRs (FP64 47 instead of 73 TFLOP/s)
                    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
                    os.path.join(HERE, "probe.hip"), "-o", tmp], check=True)
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
