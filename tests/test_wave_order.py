"""The numeric pass of the coarse products hands an accumulator in LDS from
one lane to another between two L entries.  The order of the two accesses has
to be in the program (a fence at wavefront scope), not only in what one
compiler makes of it: checked in the compiler's intermediate code."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "sci-solver_fem_amd" / "csrc"


def test_accumulators_are_fenced(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("no hipcc")
    out = tmp_path / "sparse.ll"
    subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-x", "hip",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(CSRC), "-S", "-emit-llvm",
                    str(CSRC / "sparse.hip"), "-o", str(out)], check=True, capture_output=True, timeout=120)
    body = re.search(r"^define [^\n]*num_wave_kernel.*?^}", out.read_text(), re.M | re.S).group(0)
    # the first access of every L entry of a batch
    unroll = int(re.search(r"kWaveUnroll = (\d+)", (CSRC / "sparse.hip").read_text()).group(1))
    assert len(re.findall(r'fence syncscope\("wavefront"\) acq_rel', body)) >= unroll
