"""Helpers shared by the GPU parity tests."""
import math

import numpy as np
import torch

# fp32 within 1e-5 relative, bf16/fp16 (fp32 accumulate) within 1e-2
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 1e-2}


# NHWC layers at stride 2, (N, C, H, W, K), and which of their grouped kernels deal tiles in runs: pass and element size, tile rows x
# columns
TILES_IN_RUNS = {
    (5, 256, 150, 150, 31): {"fprop 2": (5, 3), "wgrad 2": (5, 3), "fprop 4": (5, 3), "wgrad 4": (5, 3)},
    (11, 256, 290, 38, 15): {"fprop 2": (7, 1), "wgrad 2": (7, 1), "fprop 4": (7, 1), "wgrad 4": (7, 1)},
    (3, 256, 101, 301, 7): {},  # (960 tasks)
    (7, 320, 97, 130, 13): {"fprop 2": (3, 3), "wgrad 2": (3, 3), "fprop 4": (3, 3), "wgrad 4": (3, 3)},
    (17, 512, 40, 140, 31): {"fprop 2": (2, 3), "dgrad 2": (1, 2), "wgrad 2": (2, 3), "fprop 4": (2, 3), "dgrad 4": (1, 2),
                             "wgrad 4": (2, 3)},
    (8, 512, 150, 138, 31): {"fprop 2": (5, 3), "dgrad 2": (2, 2), "wgrad 2": (5, 3), "fprop 4": (5, 3)},
    (17, 256, 20, 400, 13): {"fprop 2": (1, 7), "dgrad 2": (1, 4), "wgrad 2": (1, 7), "fprop 4": (1, 7), "wgrad 4": (1, 7)},
    (11, 256, 60, 300, 7): {"fprop 2": (2, 5), "wgrad 2": (2, 5), "fprop 4": (2, 5), "wgrad 4": (2, 5)},
    (8, 256, 50, 500, 27): {"dgrad 4": (1, 4)},
}


def canonical_theta(C):
    """theta_c = (c mod 8) * 22.5 degrees, round-robin (benchmark configurations)."""
    return np.array([(c % 8) * math.pi / 8 for c in range(C)], dtype=np.float32)


def grouped_theta(C, layer_offset=0.0, n_dir=8):
    """Contiguous groups of ~C/8 channels per direction (models/convnext.py:60-77,111-114)."""
    return np.array([math.pi * ((((n_dir * (c + 1) - 1) // C) / n_dir + layer_offset) % 1)
                     for c in range(C)], dtype=np.float32)


def rel_err(got, ref):
    """Tensor-level relative errors: (max|d| / max|ref|, ||d||_2 / ||ref||_2)."""
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    d = np.abs(got - ref)
    scale = max(np.abs(ref).max(), 1e-30)
    return d.max() / scale, math.sqrt((d ** 2).sum() / max((ref ** 2).sum(), 1e-300))


def assert_close(got, ref, dtype, what=""):
    tol = TOL[dtype]
    assert got.shape == ref.shape, (what, got.shape, ref.shape)
    assert np.isfinite(np.asarray(got, dtype=np.float64)).all(), what + ": non-finite output"
    emax, el2 = rel_err(got, ref)
    assert emax <= tol and el2 <= tol, "%s: max-rel %.3e l2-rel %.3e > %.0e" % (what, emax, el2, tol)


def rounded(a, dtype):
    """Round a float32 numpy array through `dtype` (what the GPU sees), back as float32."""
    return torch.from_numpy(np.ascontiguousarray(a)).to(dtype).to(torch.float32).numpy()


def dev(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype)


def host(t):
    return t.detach().to(torch.float32).cpu().numpy()
