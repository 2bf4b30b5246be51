"""Planning of fused lm_head calls, on the CPU: fused_plan_check.cpp against the header the library itself plans with."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fused_plan") / "check")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    f"-I{os.path.join(HERE, os.pardir, 'tome_amd', 'csrc')}", os.path.join(HERE, "fused_plan_check.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_every_plan_can_be_launched_and_fits(checker, seed):
    """All selectors: a kernel form for every tile a call may take, the grid and the workspace for every number of valid tokens,
    vocab ranges that cover the vocabulary, and the token tile that the selector names."""
    run = subprocess.run([checker, str(seed)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
