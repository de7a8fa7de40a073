"""New points of a stored or hybrid plan (hm_plan_update_points): the next products are those of a
plan made of the new points, whether they are launched, captured before or captured with the
update, and the host waits for nothing."""
import numpy as np
import pytest
import torch

import hmx

pytestmark = pytest.mark.gpu


def same(a, b):
    return a.shape == b.shape and bool(((a == b) | (torch.isnan(a) & torch.isnan(b))).all())


def points(n, seed):
    x = np.sort(np.random.default_rng(seed).random(n))[::-1].copy()
    return x, x - 0.3 / n, (1.0, 0.0, 1.0, 0.0)


def dev(*vs):
    return [torch.from_numpy(v).cuda() for v in vs]


def meeting(H, x, y, rows):
    """y with some points moved onto their x, where the tree stays as it is."""
    z = y.copy()
    for i in rows:
        w = z.copy()
        w[i] = x[i]
        if np.all(np.diff(w) <= 0) and H.update_points(*dev(x, w)):
            z = w
    assert np.sum(z != y) > 0
    return z


@pytest.mark.parametrize("form", ["stored", "hybrid"])
@pytest.mark.parametrize("kernel,n,bs,r,k", [
    ("cauchykernel", 2000, 64, 15, 1), ("coulombprimekernel", 2003, 40, 9, 1),
    ("cauchykernel", 2000, 64, 15, 3), ("coulombkernel", 270001, 64, 8, 1),
    ("logkernel", 2000, 64, 15, 1)])
def test_captured_product_follows_the_points(cuda, form, kernel, n, bs, r, k):
    x, y, iv = points(n, n)
    kw = dict(blocksize=bs, rank=r, hybrid=form == "hybrid")
    H = hmx.KernelMatrix(kernel, x, y, *iv, **kw)
    b = torch.randn((n,) if k == 1 else (n, k), dtype=torch.float64, device=cuda,
                    generator=torch.Generator(device=cuda).manual_seed(2))
    first = H @ b
    out = torch.empty_like(first)
    g = H.graph(out, b)
    g.launch()
    assert same(out, first)
    on = x.copy()  # an odd rank's middle node is its cluster's center
    on[np.argmin(abs(x - 0.375))] = 0.375
    for xn, yn in ((x, meeting(H, x, y, range(3, n, max(1, n // 7)))), (on, y), (x, y)):
        ok = H.update_points(*dev(xn, yn))
        R = hmx.KernelMatrix(kernel, xn, yn, *iv, **kw)
        want = R @ b
        R.close()
        if not ok:
            continue
        out.zero_()
        g.launch()
        assert same(out, want)
        assert same(H @ b, want)
    assert same(out, first)


@pytest.mark.parametrize("transpose", [False, True])
def test_meeting_points_in_a_stored_plan(cuda, transpose):
    # infinite entries at their rows, as a plan made there reads them
    n = 3000
    x, y, iv = points(n, 4)
    H = hmx.KernelMatrix("coulombkernel", x, y, *iv, blocksize=80, rank=12)
    z = meeting(H, x, y, range(10, n, 400))
    H.update_points(*dev(x, z))
    b = torch.ones(n, dtype=torch.float64, device=cuda)
    u = (H.T @ b if transpose else H @ b).cpu().numpy()
    assert np.array_equal(np.isposinf(u), z == x) and np.isfinite(u[z != x]).all()


def test_captured_update(cuda):
    # update and product in one graph, replayed; then a launched product
    n = 4096
    x, y, iv = points(n, 7)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=64, rank=16)
    b = torch.randn(n, dtype=torch.float64, device=cuda)
    xd, yd = dev(x, y)
    out = torch.empty(n, dtype=torch.float64, device=cuda)

    def step():
        H.update_points(xd, yd, check=False)
        out.zero_()
        H.mul(out, b)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    rng = np.random.default_rng(1)
    for _ in range(3):
        xn = np.sort(x + 0.01 * (rng.random(n) - 0.5) / n)[::-1].copy()
        xd.copy_(torch.from_numpy(xn))
        g.replay()
        R = hmx.KernelMatrix("cauchykernel", xn, y, *iv, blocksize=64, rank=16)
        want = R @ b
        if H.tree_status():
            assert same(out, want) and same(H @ b, want)
        R.close()


@pytest.mark.parametrize("form", ["stored", "hybrid"])
def test_update_and_product_do_not_wait(cuda, form):
    n = 20000
    x, y, iv = points(n, 3)
    H = hmx.KernelMatrix("cauchykernel", x, y, *iv, blocksize=64, rank=16, hybrid=form == "hybrid")
    xd, yd = dev(x, y)
    b = torch.randn(n, dtype=torch.float64, device=cuda)
    u = torch.zeros_like(b)
    A = torch.randn(8192, 8192, dtype=torch.float64, device=cuda)
    C = torch.empty_like(A)
    for _ in range(2):  # the first pass also makes what later ones keep
        for _ in range(20):
            torch.mm(A, A, out=C)  # some 0.3 s queued ahead
        done = torch.cuda.Event()
        done.record()
        H.update_points(xd, yd, check=False)
        H.mul(u, b)
        waiting = not done.query()
        torch.cuda.synchronize()
    assert waiting
