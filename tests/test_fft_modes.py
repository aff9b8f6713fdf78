"""A transform pass in a mode that no kernel was built for returns an error code (it would
otherwise leave its output as it was): the dispatch, called without a GPU."""
import os
import subprocess

from codeare_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_unbuilt_modes_are_refused(cgs, tmp_path):
    lib = os.path.join(ROOT, "codeare_amd", "lib")
    out = str(tmp_path / "t_fft_modes")
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-w",
                    os.path.join(ROOT, "tests", "cpp", "t_fft_modes.cpp"), "-L", lib, "-lcgsense_hip",
                    f"-Wl,-rpath,{lib}", "-o", out], check=True)
    r = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
