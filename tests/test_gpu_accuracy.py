"""The far field's own error, against sums in extended precision: the mapped nodes are rounded (2^-53
of the point, up to 1e-12 of a deep cluster's half width), and a product must not carry that."""
import numpy as np
import pytest
import torch

import hmx

pytestmark = pytest.mark.gpu


def error(u, K, b):
    want = K @ b
    return float(np.linalg.norm((u - want).astype(np.float64)) / np.linalg.norm(want.astype(np.float64)))


@pytest.mark.parametrize("form", ["stored", "hybrid", "free"])
@pytest.mark.parametrize("kernel,n,bs,r,k,transpose,points", [
    ("cauchykernel", 1 << 20, 256, 24, 1, False, "grid"),
    ("cauchykernel", 1 << 20, 256, 24, 1, True, "grid"),
    ("logkernel", 131071, 80, 20, 4, False, "random")])
def test_float64(cuda, form, kernel, n, bs, r, k, transpose, points):
    # 2.5e-15: twice the error of the products that read U and V, which hold the basis at the
    # rounded nodes (1.3e-15 at n = 2^20)
    if points == "grid":
        x, y, iv = hmx.workloads.shifted_grid(n)
    else:
        x = np.sort(np.random.default_rng(1).random(n))[::-1].copy()
        y = x + 0.5 / n
        iv = (x[0], x[-1], y[0], y[-1])
    H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=r, hybrid=form == "hybrid",
                         matrix_free=form == "free")
    b = np.random.default_rng(2).standard_normal((n, k) if k > 1 else n)
    u = (H.T if transpose else H) @ torch.from_numpy(b).to(cuda)
    rows = np.arange(0, n, n // 32)
    out, inp = (y, x) if transpose else (x, y)
    d = out[rows].astype(np.longdouble)[:, None] - inp.astype(np.longdouble)[None, :]
    K = np.log(abs(d)) if kernel == "logkernel" else 1 / (-d if transpose else d)
    assert error(u.cpu().numpy()[rows], K, b.astype(np.longdouble)) <= 2.5e-15


@pytest.mark.parametrize("form", ["stored", "hybrid", "free"])
def test_float32(cuda, form):
    # 1e-6: sixteen roundings (the basis at the exact nodes with F at the rounded ones: 7.8e-6).
    # A Float32 point meets a node here and there: those rows of a stored product are NaN.
    n = 500009
    x, y, iv = hmx.workloads.shifted_grid(n)
    x, y = x.astype(np.float32), y.astype(np.float32)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=40, rank=10, hybrid=form == "hybrid",
                         matrix_free=form == "free")
    b = np.random.default_rng(2).standard_normal(n).astype(np.float32)
    u = (H @ torch.from_numpy(b).to(cuda)).cpu().numpy()
    rows = np.arange(0, n, n // 256)
    rows = rows[np.isfinite(u[rows])]
    assert len(rows) > 16 and (form == "stored" or np.isfinite(u).all())
    K = 1 / (x[rows].astype(np.float64)[:, None] - y.astype(np.float64)[None, :])
    assert error(u[rows], K, b.astype(np.float64)) <= 1e-6


@pytest.mark.parametrize("form", ["hybrid", "free"])
@pytest.mark.parametrize("seed", [2, 3])
def test_deep_nested(cuda, form, seed):
    # eight right-hand sides over trees whose halves are rounded by more than 1e-12: no further off
    # than the products that apply every covering cluster (4.4e-15)
    n, k = 400000, 8
    x = np.sort(np.random.default_rng(seed).random(n))[::-1].copy()
    y = x + 0.5 / n
    H = hmx.KernelMatrix("logkernel", x, y, x[0], x[-1], y[0], y[-1], blocksize=40, rank=24,
                         hybrid=form == "hybrid", matrix_free=form == "free")
    assert H.info["nested"] == 1
    b = np.random.default_rng(100 + seed).standard_normal((n, k))
    rows = np.arange(0, n, n // 48)
    u = H.matvec(torch.from_numpy(b).to(cuda), mfma=True).cpu().numpy()[rows]
    K = np.log(abs(x[rows].astype(np.longdouble)[:, None] - y.astype(np.longdouble)[None, :]))
    assert error(u, K, b.astype(np.longdouble)) <= 4.4e-15
