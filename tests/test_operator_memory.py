"""The host side of the operator's build with little device memory (tests/host/operator_memory.cpp): spmm.hip
compiled for the CPU against stand-ins for the HIP runtime and the kernels.  CPU only."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "fastdose_amd" / "csrc"
ROCM = Path("/opt/rocm/include")


@pytest.mark.skipif(shutil.which("g++") is None or not (ROCM / "hip" / "hip_runtime.h").exists(),
                    reason="needs g++ and the HIP headers")
def test_operator_is_built_wherever_the_general_path_fits(tmp_path):
    exe = tmp_path / "operator_memory"
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}", f"-I{ROOT / 'include'}", f"-I{CSRC}",
           "-x", "c++", str(ROOT / "tests" / "host" / "operator_memory.cpp"), str(CSRC / "spmm.hip"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "operator memory: ok" in run.stdout, run.stdout[-4000:] + run.stderr[-2000:]
