"""Products are linear in their input over the element type's range: inputs and points scaled by
powers of two, where no term of the sum leaves the range, give the scaled result."""
import numpy as np
import pytest
import torch

import hmx
import oracle as O

pytestmark = pytest.mark.gpu

KID = {"cauchykernel": O.CAUCHY, "coulombkernel": O.COULOMB, "coulombprimekernel": O.COULOMB3}
SIGN = {"cauchykernel": -1.0, "coulombkernel": 1.0, "coulombprimekernel": -1.0}


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# exponents of the points' and the inputs' scale
@pytest.mark.parametrize("dtype,kernel,pe,be", [
    ("f32", "cauchykernel", 0, -93), ("f32", "cauchykernel", 0, 80),
    ("f32", "cauchykernel", -21, -53), ("f32", "cauchykernel", -21, -60),   # spacing 1e-9
    ("f32", "cauchykernel", 36, 50), ("f32", "coulombkernel", -21, -80),    # spacing 1e8, 1e-9
    ("f32", "coulombprimekernel", 0, -90), ("f32", "coulombprimekernel", 9, 60),
    ("f64", "cauchykernel", 0, -980), ("f64", "cauchykernel", 0, 900),
    ("f64", "coulombkernel", -120, -500), ("f64", "coulombprimekernel", -100, -200),
    ("f64", "coulombprimekernel", 100, 200)])
@pytest.mark.parametrize("transpose", [False, True])
def test_scaled_inputs(cuda, dtype, kernel, pe, be, transpose):
    # against the oracle's mul! at an input of order one, scaled (exactly): the products' bars,
    # 1e-12 in Float64 and 1e-5 in Float32
    n, bs, r = 700, 40, 10
    f32 = dtype == "f32"
    dt = np.float32 if f32 else np.float64
    i = np.arange(n, 0, -1, dtype=np.float64)
    ps = 2.0 ** pe
    x, y = ((i - 0.25) / n * ps).astype(dt), ((i - 0.75) / n * ps).astype(dt)
    iv = (ps, 0.0, ps, 0.0)
    b = np.random.default_rng(3).standard_normal(n).astype(dt)
    if transpose:  # H(x, y)' = s H(y, x)
        ref = SIGN[kernel] * O.Tree(KID[kernel], y, x, *iv, bs, r, f32=f32).matvec(b)
    else:
        ref = O.Tree(KID[kernel], x, y, *iv, bs, r, f32=f32).matvec(b)
    H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=r, matrix_free=True)
    v = torch.from_numpy(b * dt(2.0 ** be)).to(cuda)
    u = (H.T @ v if transpose else H @ v).cpu().numpy()
    assert rel(u.astype(np.float64) * 2.0 ** -be, ref) <= (1e-5 if f32 else 1e-12)


@pytest.mark.parametrize("transpose", [False, True])
def test_scaled_inputs_units(cuda, transpose):
    # more than 4096 chunks (columns through LDS): the scaled product against the product
    n = 1 << 20
    x, y, iv = hmx.workloads.shifted_grid(n)
    H = hmx.KernelMatrix("cauchykernel", x.astype(np.float32), y.astype(np.float32), *iv,
                         blocksize=64, rank=16, matrix_free=True)
    b = torch.randn(n, dtype=torch.float32, device=cuda,
                    generator=torch.Generator(device=cuda).manual_seed(5))
    op = H.T if transpose else H
    want = (op @ b).cpu().numpy()
    for e in (-93, 70):
        got = (op @ (b * 2.0 ** e)).cpu().numpy()
        assert rel(got.astype(np.float64) * 2.0 ** -e, want) <= 1e-5


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("form", ["hybrid", "free"])
@pytest.mark.parametrize("k", [1, 3, 8])
@pytest.mark.parametrize("rank", [20, 32])
def test_top_of_the_range(cuda, dtype, form, k, rank):
    # results in the last binary order below the largest number, and nothing on the way beyond it:
    # a power of two times the product at order one
    n = 700
    dt = np.float32 if dtype == "f32" else np.float64
    i = np.arange(n, 0, -1, dtype=np.float64)
    x, y = ((i - 0.25) / n).astype(dt), ((i - 0.75) / n).astype(dt)
    H = hmx.KernelMatrix("cauchykernel", x, y, 1.0, 0.0, 1.0, 0.0, blocksize=40, rank=rank,
                         hybrid=form == "hybrid", matrix_free=form == "free")
    b = torch.from_numpy(np.abs(np.random.default_rng(3).standard_normal((n, k))).astype(dt)).to(cuda)
    b = b[:, 0].contiguous() if k == 1 else b
    for op in (H, H.T):
        want = (op @ b).cpu().numpy().astype(np.float64)
        e = int(np.floor(np.log2(float(np.finfo(dt).max)) - np.log2(np.abs(want).max())))
        got = (op @ (b * 2.0 ** e)).cpu().numpy().astype(np.float64)
        assert rel(got * 2.0 ** -e, want) <= (1e-5 if dtype == "f32" else 1e-12)
