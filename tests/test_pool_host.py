"""The device memory pool over a stub of the HIP runtime (no GPU): reuse, waiting,
stream capture, its bound and failed allocations (tests/pool_driver.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "ra-spmm_amd" / "csrc"


def test_pool_over_a_stub_runtime(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None or not Path("/opt/rocm/include/hip/hip_runtime_api.h").exists():
        pytest.skip("needs g++ and the HIP headers")
    exe = tmp_path / "pool"
    cmd = [gxx, "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
           f"-I{CSRC}", str(Path(__file__).with_name("pool_driver.cpp")), str(CSRC / "common.cpp"), "-lpthread", "-o", str(exe)]
    build = subprocess.run(cmd, capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr
