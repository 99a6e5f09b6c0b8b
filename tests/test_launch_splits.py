"""CPU-only: the host code that cuts the window, grouped and product kernels' launches, compiled by itself and checked over
the shapes that it accepts (tests/host)."""
import os
import subprocess

import pytest

from oriented1d_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("program", ["window_units", "grouped_tasks", "linear_splits"])
def test_launch_splits(program, tmp_path):
    exe = str(tmp_path / program)
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + build.CSRC,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", program + ".cpp"),
                    "-o", exe], check=True)
    done = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout


def test_product_and_tail_launches_stay_below_two_to_the_32_threads():
    """The rules in front of the product kernels and the block's tail against their grids (dwo_linear.h, dwo_block.hip)."""
    import random

    import torch

    from oriented1d_amd import fused
    rng = random.Random(0)
    for _ in range(4000):
        N, K = 8 * rng.choice([1, 2, 3, 8, 12, 15, 16, 17, 32, 33, 48, 512, 8192]), 8 * rng.choice([1, 2, 12, 128])
        most = min((fused._PRODUCT_MAX - 1) // K, (1 << 37) // N)  # (2^37 outputs: 275 GB)
        rows = rng.choice([most, rng.randint(1, most)])
        mtiles = -(-rows // 128)
        for nt in {96, 128} if N % 96 == 0 else {128}:
            assert -(-mtiles // 8) * 8 * -(-N // nt) * 256 < 1 << 32, (rows, N)
    for shape in ((1 << 24, 1, 1, 8), ((1 << 24) - 1, 1, 1, 8), (1 << 20, 9, 9, 24), (1 << 22, 2, 2, 72), (64, 56, 56, 128), (0, 7, 7, 8)):
        y = torch.empty(shape, device="meta")
        if fused._tail_covers(y):
            N, H, W, C = shape
            assert N * -(-H * W // 64) * -(-C // 64) * 256 < 1 << 32, shape
    assert not fused._tail_covers(torch.empty(1 << 24, 1, 1, 8, device="meta"))
    assert fused._tail_covers(torch.empty(64, 56, 56, 128, device="meta"))
