"""Sizes and right-hand-side counts at which products over the interval trees change their form."""
import numpy as np
import pytest
import torch

import hmx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,form", [("cauchykernel", "free"), ("cauchykernel", "hybrid"),
                                         ("logkernel", "free"), ("logkernel", "stored")])
@pytest.mark.parametrize("n", [65472, 65537, 65700])
@pytest.mark.parametrize("k", [1, 3])
def test_chunks_and_units(cuda, kernel, form, n, k):
    # 1024 chunks (log kernel 4096) of 64 rows or less: a workgroup of the near field takes a chunk;
    # above, a wavefront takes two. 1e-12: the products' bar against dense rows
    x = np.sort(np.random.default_rng(n).random(n))[::-1].copy()
    y = x + 0.5 / n
    H = hmx.KernelMatrix(kernel, x, y, x[0], x[-1], y[0], y[-1], blocksize=80, rank=20,
                         hybrid=form == "hybrid", matrix_free=form == "free")
    b = torch.randn((n, k) if k > 1 else n, dtype=torch.float64, device=cuda)
    rows = torch.arange(0, n, 211, device=cuda)
    xd, yd = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    for u, d in ((H @ b, xd[rows][:, None] - yd[None, :]), (H.T @ b, xd[None, :] - yd[rows][:, None])):
        K = d.abs().log() if kernel == "logkernel" else 1 / d
        assert ((u[rows] - K @ b).norm() / (K @ b).norm()).item() <= 1e-12


@pytest.mark.parametrize("n", [1000, 4096, 4500])
@pytest.mark.parametrize("k", [7, 8, 13, 16])
def test_eight_float32(cuda, n, k):
    # up to 128 chunks a stored Float32 plan takes eight right-hand sides per level, the rest over
    # the trees: each column against dense rows, Float32's bar of 1e-5
    x, y, iv = hmx.workloads.shifted_grid(n)
    x, y = x.astype(np.float32), y.astype(np.float32)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=40, rank=10)
    b = torch.randn(n, k, dtype=torch.float32, device=cuda)
    u = (H @ b).double()
    ok = torch.isfinite(u).all(1)
    assert ok.sum().item() > n // 2
    xd, yd = (torch.from_numpy(v.astype(np.float64)).to(cuda) for v in (x, y))
    ref = (1 / (xd[ok][:, None] - yd[None, :])) @ b.double()
    assert ((u[ok] - ref).norm(dim=0) / ref.norm(dim=0)).max().item() <= 1e-5
