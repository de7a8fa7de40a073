"""Points of x equal to points of y: the infinite entries stay at their rows."""
import numpy as np
import pytest
import torch

import hmx

pytestmark = pytest.mark.gpu


def coincident(n, step, seed):
    """Every step-th y is its x: one infinite entry in each of these rows and columns."""
    x = np.sort(np.random.default_rng(seed).random(n))[::-1].copy()
    y = 0.5 * (x + np.append(x[1:], 2 * x[-1] - x[-2]))
    at = np.arange(0, n, step)
    y[at] = x[at]
    return x, y, (x[0], x[-1], y[0], y[-1]), at


@pytest.mark.parametrize("kernel,k", [("logkernel", 1), ("logkernel", 3), ("cauchykernel", 1),
                                      ("coulombprimekernel", 1)])
@pytest.mark.parametrize("n,bs", [(300, 80), (1000, 24), (1003, 80), (300007, 64)])
@pytest.mark.parametrize("transpose", [False, True])
def test_matrix_free_infinite_entries(cuda, kernel, k, n, bs, transpose):
    # a wavefront's last columns of a block are padded with repeated ones at weight zero:
    # 0 * inf there would turn the row's infinity into NaN
    x, y, iv, at = coincident(n, 7, n)
    H = hmx.KernelMatrix(kernel, x, y, *iv, blocksize=bs, rank=12, matrix_free=True)
    b = torch.ones(n, dtype=torch.float64, device=cuda) if k == 1 else \
        torch.ones(n, k, dtype=torch.float64, device=cuda)
    u = (H.T @ b if transpose else H @ b).cpu().numpy()
    want = np.zeros(n, bool)
    want[at] = True
    for q in range(k):
        c = u if k == 1 else u[:, q]
        assert np.array_equal(np.isinf(c), want) and np.isfinite(c[~want]).all()
