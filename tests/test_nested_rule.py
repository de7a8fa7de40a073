"""The nested far field's rule: halves of intervals whose ends are rounded still count as halves."""
import numpy as np
import pytest

import hmx


def _points(n, seed, shift=0.0):
    x = np.sort(np.random.default_rng(seed).random(n))[::-1] + shift
    y = x + 0.5 / n
    return x, y, (x[0], x[-1], y[0], y[-1])


@pytest.mark.parametrize("seed", range(6))
def test_deep_random_intervals_nest(seed):
    # depth >= 14 of intervals with arbitrary ends: the centers are rounded to
    # 2^-53, 2^-38 of the deepest halfwidths
    x, y, iv = _points(400000, seed)
    H = hmx.KernelMatrix("logkernel", x, y, *iv, blocksize=40, rank=8, tree_only=True)
    i = H.info
    assert i["depth"] >= 14 and i["nested"] == 1


def test_intervals_far_from_zero_do_not_nest():
    # at 1e6 the centers' rounding is 1e-6 of the deepest halfwidths: per-level far field
    x, y, iv = _points(40000, 1, shift=1e6)
    H = hmx.KernelMatrix("logkernel", x, y, *iv, blocksize=40, rank=8, tree_only=True)
    assert H.info["nested"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [2, 3])
def test_deep_nested_product(cuda, seed):
    # 1e-12: rank 24 interpolates the far blocks to rounding, and depth 14
    # leaves 2^-53 * 2^14 = 2e-12 of a halfwidth at the deepest blocks, whose
    # share of a row's sum is below a tenth
    import torch
    n, k = 400000, 8
    x, y, iv = _points(n, seed)
    H = hmx.KernelMatrix("logkernel", x, y, *iv, blocksize=40, rank=24, hybrid=True)
    assert H.info["nested"] == 1
    b = torch.randn(n, k, dtype=torch.float64, device=cuda)
    u = H.matvec(b, mfma=True)
    rows = np.random.default_rng(seed).integers(0, n, 200)
    d = torch.from_numpy(x[rows]).to(cuda)[:, None] - torch.from_numpy(y).to(cuda)[None, :]
    ref = d.abs().log() @ b
    err = (u[torch.from_numpy(rows).to(cuda)] - ref).norm() / ref.norm()
    assert err.item() <= 1e-12
