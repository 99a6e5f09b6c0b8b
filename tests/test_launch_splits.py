"""CPU-only: the host code that cuts the window, grouped and product kernels' launches, compiled by itself and checked over
the shapes that it accepts (tests/host)."""
import os
import subprocess

import pytest

from parity_util import TILES_IN_RUNS

from oriented1d_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _compiled(program, folder):
    exe = str(folder / program)
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + build.CSRC,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", program + ".cpp"),
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("program", ["window_units", "grouped_tasks", "grouped_runs", "linear_splits"])
def test_launch_splits(program, tmp_path):
    done = subprocess.run([_compiled(program, tmp_path)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout


@pytest.fixture(scope="module")
def grouped_runs(tmp_path_factory):
    return _compiled("grouped_runs", tmp_path_factory.mktemp("host"))


def test_shapes_whose_tiles_go_in_runs(grouped_runs):
    """The layers that the GPU tests take for this reach it: every pass and element size, each with the tile columns that are stated."""
    seen = set()
    for shape, want in TILES_IN_RUNS.items():
        got = {}
        for line in subprocess.run([grouped_runs, *map(str, shape)], stdout=subprocess.PIPE, text=True, check=True).stdout.splitlines():
            name, size, run, rows, columns = line.split()
            if int(run) > 0:
                got[name + " " + size] = (int(rows), int(columns))
        assert got == want, shape
        seen.update((k, columns) for k, (_, columns) in got.items())
    for size in ("2", "4"):
        assert {("fprop " + size, c) for c in (1, 3, 5, 7)} | {("wgrad " + size, c) for c in (1, 3, 5, 7)} <= seen
        assert {("dgrad " + size, c) for c in (2, 4)} <= seen


@pytest.mark.parametrize("layer,runs", [
    # x and y of 253 and 260 MB, or far more: K = 31 everywhere, smaller kernels by pass and type; three tile columns of dgrad;
    # many channels; few tasks
    ((64, 64, 224, 224, 31), {"fprop 2", "dgrad 2", "wgrad 2", "fprop 4", "dgrad 4", "wgrad 4"}),
    ((64, 64, 224, 224, 15), {"dgrad 2", "wgrad 2"}), ((64, 64, 224, 224, 7), {"dgrad 2"}),
    ((33, 64, 224, 224, 7), {"fprop 2", "wgrad 2"}), ((34, 64, 224, 224, 7), set()),
    ((34, 64, 320, 288, 31), {"fprop 2", "wgrad 2", "fprop 4", "wgrad 4"}), ((8, 64, 512, 512, 31), {"dgrad 4"}),
    ((128, 128, 112, 112, 31), {"fprop 2", "wgrad 2", "fprop 4"}), ((40, 192, 224, 224, 31), {"fprop 2", "wgrad 2", "fprop 4"}),
    ((40, 256, 224, 224, 31), {"fprop 2", "fprop 4"}),
    ((16, 128, 224, 224, 15), {"fprop 2", "wgrad 2"}), ((3, 64, 200, 300, 31), set())])
def test_rule_for_tiles_in_runs(layer, runs, grouped_runs):
    out = subprocess.run([grouped_runs, *map(str, layer)], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert {" ".join(l.split()[:2]) for l in out.splitlines() if int(l.split()[2]) > 0} == runs


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
