"""Host loops behind the C ABI that run in shares on threads (the tables a trajectory is
laid out in): every share runs once also where threads cannot be started, and what a share
throws reaches the caller, whose entry point returns it as an error code."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("cpp") / "t_host_threads")
    subprocess.run([gxx, "-O1", "-std=c++17", "-Wall", "-Werror", os.path.join(ROOT, "tests", "cpp", "t_host_threads.cpp"),
                    "-pthread", "-ldl", "-o", out], check=True)
    return out


@pytest.mark.parametrize("shares,allowed,thrower", [
    (0, 0, -1), (1, 0, -1), (1, 0, 0), (16, 15, -1), (16, 0, -1), (16, 3, -1), (16, 15, 0), (16, 15, 7), (16, 3, 9), (16, 3, 2),
])
def test_shares(program, shares, allowed, thrower):
    r = subprocess.run([program, str(shares), str(allowed), str(thrower)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == [str(shares), "1" if thrower >= 0 else "0"]


def test_no_bare_threads_behind_the_abi():
    """std::thread only inside the helper: elsewhere an exception would end the process."""
    src = os.path.join(ROOT, "codeare_amd", "csrc")
    users = [f for f in os.listdir(src) if f.endswith((".hip", ".hpp")) and f != "host_threads.hpp"
             and "std::vector<std::thread>" in open(os.path.join(src, f)).read()]
    assert users == []
