"""CPU-only: the host code that cuts the window kernels' launches, compiled by itself and checked over the
shapes that it accepts (tests/host/window_units.cpp)."""
import os
import subprocess

from oriented1d_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_window_units(tmp_path):
    exe = str(tmp_path / "window_units")
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + build.CSRC,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", "window_units.cpp"),
                    "-o", exe], check=True)
    done = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout
