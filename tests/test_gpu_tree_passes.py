"""Single right-hand sides over the interval trees (nested1.h): sizes where the passes change
shape, against the oracle's mul! (same tree and rank, so only rounding differs: the products' bar
of 1e-12), dense rows, and the stored-entry route they replace."""
import math

import numpy as np
import pytest
import torch

import hmx
import oracle as O

pytestmark = pytest.mark.gpu

KID = {"cauchykernel": O.CAUCHY, "coulombkernel": O.COULOMB,
       "coulombprimekernel": O.COULOMB3, "logkernel": O.LOG}
# f(x, y) = s f(y, x)
SIGN = {"cauchykernel": -1.0, "coulombkernel": 1.0, "coulombprimekernel": -1.0, "logkernel": 1.0}


def points(n, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "random":
        x = np.sort(rng.random(n))[::-1].copy()
        y = x + 0.5 / n
    else:  # geometric: depth beyond 40, long paths above the subtrees, empty halves
        x = np.sort(2.0 ** (-np.arange(n) * 50.0 / n) * (1 + 1e-4 * rng.random(n)))[::-1].copy()
        y = x * (1 - 5.0 / n)
    return x, y, (x[0], x[-1], y[0], y[-1])


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("kernel", list(KID))
@pytest.mark.parametrize("n,kind,bs,r", [
    (1, "random", 8, 4), (63, "random", 80, 20), (65, "random", 80, 20),   # no far field
    (160, "random", 80, 20),                                               # one subtree, no path
    (700, "random", 16, 1), (700, "random", 16, 2), (700, "random", 24, 7),  # rank buckets' edges
    (900, "random", 40, 8), (900, "random", 40, 9), (900, "random", 64, 16),
    (900, "random", 64, 17), (1500, "random", 96, 25), (1500, "random", 130, 32),
    (1500, "random", 130, 33),                                             # the per-level passes
    (3001, "random", 300, 24),                                             # leaves of several chunks
    (2000, "geometric", 40, 16), (3000, "geometric", 12, 10)])
def test_products_vs_oracle(cuda, kernel, n, kind, bs, r):
    x, y, iv = points(n, kind, n + r)
    rng = np.random.default_rng(1)
    b, c = rng.standard_normal(n), rng.standard_normal(n)
    if n == 1:
        iv = (1.0, 0.0, 1.0, 0.0)
    ref = O.Tree(KID[kernel], x, y, *iv, bs, r).matvec(b)
    # H(x, y)' = s H(y, x): the block tree of the exchanged points
    reft = SIGN[kernel] * O.Tree(KID[kernel], y, x, iv[2], iv[3], iv[0], iv[1], bs, r).matvec(c)
    bd, cd = torch.from_numpy(b).to(cuda), torch.from_numpy(c).to(cuda)
    for form in ("stored", "hybrid", "free"):
        H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=r, hybrid=form == "hybrid",
                             matrix_free=form == "free")
        assert rel((H @ bd).cpu().numpy(), ref) <= 1e-12, form
        assert rel((H.T @ cd).cpu().numpy(), reft) <= 1e-12, form
        # accumulating, strided, at an offset
        u = torch.ones(2 * n + 3, dtype=torch.float64, device=cuda)
        v = torch.zeros(3 * n + 5, dtype=torch.float64, device=cuda)
        v[1::3][:n] = bd
        H.mul(u, v, 3, 2, 3, 2)
        assert rel(u[2::2][:n].cpu().numpy() - 1, ref) <= 1e-12 * (1 + 1 / np.linalg.norm(ref) * n), form
        H.close()


@pytest.mark.parametrize("n,bs,r", [(262143, 80, 20), (263000, 80, 20), (300001, 512, 32)])
@pytest.mark.parametrize("transpose", [False, True])
def test_units_and_chunks(cuda, n, bs, r, transpose):
    # 4096 chunks: below, a workgroup of the near field takes a chunk; above, a
    # wavefront takes two. 1e-12: the n = 2^20 products' bar against dense rows
    x, y, iv = points(n, "random", 3)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=bs, rank=r, matrix_free=True)
    b = torch.randn(n, dtype=torch.float64, device=cuda)
    u = H.T @ b if transpose else H @ b
    rows = torch.arange(0, n, 997, device=cuda)
    xd, yd = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    d = xd[None, :] - yd[rows][:, None] if transpose else xd[rows][:, None] - yd[None, :]
    ref = (1.0 / d) @ b
    assert ((u[rows] - ref).norm() / ref.norm()).item() <= 1e-12
    # the same sums whatever the order of launches around it
    assert torch.equal(u, H.T @ b if transpose else H @ b)


@pytest.mark.parametrize("form", ["stored", "hybrid"])
def test_coincident_points_keep_stored_entries(cuda, form):
    # a point of x equal to one of y: the stored entry is infinite, as the
    # reference's, and the product reads it
    x, y, iv = points(1000, "random", 5)
    y = y.copy()
    y[500] = x[500]
    y = np.sort(y)[::-1].copy()
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=80, rank=20, hybrid=form == "hybrid")
    assert H.info["nonfinite"] == 1
    b = torch.ones(1000, dtype=torch.float64, device=cuda)
    u = H @ b
    assert torch.isinf(u).sum().item() == 1 and torch.isfinite(u).sum().item() == 999


def test_moved_points_and_user_entries(cuda):
    # new points: the stored forms read the re-formed entries
    n = 4096
    w = hmx.workloads.config_plain(n=n, blocksize=64, rank=16)
    x2, y2 = w["x"] + 0.05 / n, w["y"] - 0.03 / n
    b = torch.from_numpy(w["b"]).to(cuda)
    ref = O.Tree(O.CAUCHY, x2, y2, *w["intervals"], 64, 16).matvec(w["b"])
    for form in ("stored", "hybrid", "free"):
        H = hmx.KernelMatrix("cauchykernel", w["x"], w["y"], *w["intervals"], blocksize=64, rank=16,
                             hybrid=form == "hybrid", matrix_free=form == "free")
        assert H.update_points(torch.from_numpy(x2).to(cuda), torch.from_numpy(y2).to(cuda))
        assert rel((H @ b).cpu().numpy(), ref) <= 1e-12, form
    # a caller's own f: its entries, not 1/(x - y), are applied
    H = hmx.KernelMatrix(lambda s, t: 3.0 / (s - t), w["x"], w["y"], *w["intervals"], blocksize=64,
                         rank=16, hybrid=True)
    ref = 3.0 * O.Tree(O.CAUCHY, w["x"], w["y"], *w["intervals"], 64, 16).matvec(w["b"])
    assert rel((H @ b).cpu().numpy(), ref) <= 1e-12


@pytest.mark.parametrize("scale", [1e-80, 1e-60, 1e60, 1e90, 1e110])
@pytest.mark.parametrize("kernel", ["cauchykernel", "coulombkernel", "coulombprimekernel"])
def test_scaled_points(cuda, kernel, scale):
    # products of four d^m leave the double range at these scales: the terms
    # are then formed one by one (stored: the entries are read where they are
    # beyond it)
    n = 600
    x, y, iv = points(n, "random", 9)
    p = KID[kernel] + 1
    x, y, iv = x * scale, y * scale, tuple(v * scale for v in iv)
    if abs(p * math.log10(scale)) >= 300:
        pytest.skip("the entries themselves leave the range")
    b = np.random.default_rng(2).standard_normal(n)
    ref = O.Tree(KID[kernel], x, y, *iv, 40, 16).matvec(b)
    for form in ("stored", "free"):
        H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=40, rank=16, matrix_free=form == "free")
        u = (H @ torch.from_numpy(b).to(cuda)).cpu().numpy()
        assert np.isfinite(u).all() and rel(u / np.abs(ref).max(), ref / np.abs(ref).max()) <= 1e-12


@pytest.mark.parametrize("n,bs,r", [(500, 40, 10), (30000, 40, 10)])
def test_float32(cuda, n, bs, r):
    # Float32 products: 1e-5 of the Float32 oracle's mul! (its own bar)
    x, y, iv = hmx.workloads.shifted_grid(n)
    x, y = x.astype(np.float32), y.astype(np.float32)
    b = np.random.default_rng(4).standard_normal(n).astype(np.float32)
    ref = O.Tree(O.CAUCHY, x, y, *iv, bs, r, f32=True).matvec(b)
    for form in ("hybrid", "free"):
        H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=bs, rank=r,
                             hybrid=form == "hybrid", matrix_free=form == "free")
        u = (H @ torch.from_numpy(b).to(cuda)).cpu().numpy()
        assert rel(u.astype(np.float64), ref.astype(np.float64)) <= 1e-5


@pytest.mark.parametrize("transpose", [False, True])
def test_float32_units(cuda, transpose):
    # more than 4096 chunks; the oracle's own factors are not finite here (nodes
    # meet points), so against dense rows, within the Float32 oracle's 2e-5
    n = 300000
    x, y, iv = hmx.workloads.shifted_grid(n)
    x, y = x.astype(np.float32), y.astype(np.float32)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=64, rank=16, hybrid=True)
    b = torch.randn(n, dtype=torch.float32, device=cuda)
    u = H.T @ b if transpose else H @ b
    rows = torch.arange(0, n, 499, device=cuda)
    xd, yd = (torch.from_numpy(v.astype(np.float64)).to(cuda) for v in (x, y))
    d = xd[None, :] - yd[rows][:, None] if transpose else xd[rows][:, None] - yd[None, :]
    ref = (1.0 / d) @ b.double()
    assert ((u[rows].double() - ref).norm() / ref.norm()).item() <= 2e-5


def test_moved_onto_a_node(cuda):
    # odd rank: a cluster's middle node is its center. A stored plan moved onto
    # one has non-finite U, as a plan built there has, and its product is not
    # finite; moved off again it is
    n, kw = 2000, dict(blocksize=64, rank=15)
    x, y, _ = points(n, "random", 11)
    iv = (1.0, 0.0, 1.0, 0.0)
    on = x.copy()
    on[np.argmin(abs(x - 0.375))] = 0.375
    b = torch.ones(n, dtype=torch.float64, device=cuda)
    R = hmx.KernelMatrix("cauchykernel", on, y, *iv, **kw)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, **kw)
    assert R.info["nonfinite"] > 0 and H.info["nonfinite"] == 0
    u0 = H @ b
    xd, od, yd = (torch.from_numpy(v).to(cuda) for v in (x, on, y))
    H.update_points(od, yd)
    want = R @ b
    assert not torch.isfinite(want).all()
    assert torch.equal(torch.isfinite(H @ b), torch.isfinite(want))
    H.update_points(xd, yd)
    assert torch.equal(H @ b, u0)


@pytest.mark.parametrize("kernel", ["coulombkernel", "logkernel"])
@pytest.mark.parametrize("n,bs,r", [(50, 80, 20), (900, 40, 9), (1500, 130, 32), (2501, 80, 20)])
@pytest.mark.parametrize("k", [2, 3, 4, 5, 7])
def test_several_rhs(cuda, kernel, n, bs, r, k):
    # up to four right-hand sides per launch, rows or columns contiguous, accumulating; each column
    # within the products' 1e-12 of the oracle's mul!
    x, y, iv = points(n, "random", n)
    B = np.random.default_rng(k).standard_normal((n, k))
    t = O.Tree(KID[kernel], x, y, *iv, bs, r)
    tt = O.Tree(KID[kernel], y, x, iv[2], iv[3], iv[0], iv[1], bs, r)
    ref = np.stack([t.matvec(np.ascontiguousarray(B[:, q])) for q in range(k)], 1)
    reft = SIGN[kernel] * np.stack([tt.matvec(np.ascontiguousarray(B[:, q])) for q in range(k)], 1)
    Bd = torch.from_numpy(B).to(cuda)
    Bc = Bd.t().contiguous().t()
    for form in ("stored", "free"):
        H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=r, matrix_free=form == "free")
        for b in (Bd, Bc):
            u, v = (H @ b).cpu().numpy(), (H.T @ b).cpu().numpy()
            for q in range(k):
                assert rel(u[:, q], ref[:, q]) <= 1e-12 and rel(v[:, q], reft[:, q]) <= 1e-12, (form, q)
        u = Bd.clone()
        H.mul(u, Bd)
        assert rel(u.cpu().numpy(), ref + B) <= 1e-12
        H.close()


@pytest.mark.parametrize("kernel", ["cauchykernel", "logkernel"])
@pytest.mark.parametrize("form", ["stored", "free"])
def test_several_rhs_units(cuda, kernel, form):
    # more than 4096 chunks, against the same plan's single products (rounding
    # of another summation order: the per-column bar of the multi-RHS passes, 1e-13)
    n = 270001
    x, y, iv = points(n, "random", 8)
    H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=80, rank=16, matrix_free=form == "free")
    B = torch.randn(n, 3, dtype=torch.float64, device=cuda)
    u, v = H @ B, H.T @ B
    for q in range(3):
        b = B[:, q].contiguous()
        assert ((u[:, q] - H @ b).norm() / u[:, q].norm()).item() <= 1e-13
        assert ((v[:, q] - H.T @ b).norm() / v[:, q].norm()).item() <= 1e-13


@pytest.mark.parametrize("kernel", ["cauchykernel", "coulombkernel", "coulombprimekernel", "logkernel"])
@pytest.mark.parametrize("n,bs,r", [(50, 80, 20), (900, 40, 9), (2501, 64, 16), (40001, 64, 32)])
def test_gradient_chain(cuda, kernel, n, bs, r):
    # the gradient passes' far field over the trees, both directions, against the
    # matrix-free products (the same terms, summed in another order: 1e-13)
    x, y, iv = points(n, "random", n)
    H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=r, matrix_free=True)
    g = torch.Generator(device=cuda).manual_seed(n)
    b, q = (torch.randn(n, dtype=torch.float64, device=cuda, generator=g) for _ in range(2))
    u, _ = H.matvec_grad(b)
    gb, _ = H.tgrad(q, b)
    for got, want in ((u, H @ b), (gb, H.T @ q)):
        assert ((got - want).norm() / want.norm()).item() <= 1e-13
