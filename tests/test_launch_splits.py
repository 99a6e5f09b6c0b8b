"""CPU-only: the host code that cuts the window and grouped kernels' launches, compiled by itself and checked over
the shapes that it accepts (tests/host)."""
import os
import subprocess

import pytest

from oriented1d_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("program", ["window_units", "grouped_tasks"])
def test_launch_splits(program, tmp_path):
    exe = str(tmp_path / program)
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + build.CSRC,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", program + ".cpp"),
                    "-o", exe], check=True)
    done = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout
