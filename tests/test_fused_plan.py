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


def test_planning_stays_off_the_clock(checker):
    """A call's planning on the host (best of 200 runs, so a busy machine does not count): 0.2 - 0.3 us up to 8192 tokens and 3 beyond,
    where walking every number of token tiles took 1.8, 3.5, 117 and 797."""
    out = subprocess.run([checker, "time", "200", "4096", "16384", "65536"], capture_output=True, text=True, check=True).stdout
    took = {int(n): float(us) for n, us in (line.split() for line in out.splitlines())}
    for n, most in ((200, 1.2), (4096, 1.2), (16384, 30.0), (65536, 60.0)):
        assert took[n] < most, took
