"""The device-memory pool on the CPU, over a simulated device (devpool_host.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "sci-solver_fem_amd" / "csrc"
ROCM = Path("/opt/rocm/include")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx or not ROCM.exists():
        pytest.skip("no g++ or HIP headers")
    exe = tmp_path_factory.mktemp("devpool") / "devpool"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", str(ROCM), "-I", str(CSRC),
                    str(HERE / "devpool_host.cpp"), str(CSRC / "devpool.cpp"), "-o", str(exe), "-pthread"],
                   check=True, timeout=120)
    return exe


@pytest.mark.parametrize("scenario", ["foreign_work", "failed_allocation", "reserve_ages", "flush_beside_work"])
def test_devpool(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
