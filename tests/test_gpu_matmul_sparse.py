"""Products of operands with many zeros: no further from 64 bits than fp32
multiply-adds, one rounding per nonzero product, on every tile (gemm_tile.h),
and the same bits for the same row wherever it stands in a tile.
"""
import numpy as np
import pytest

import gpu_util as U

pytestmark = pytest.mark.gpu


def _fma(a, b):
    """a @ b with one float32 rounding per k (an addition of +-0 rounds nothing)."""
    acc = np.zeros((a.shape[0], b.shape[1]), np.float32)
    for k in range(a.shape[1]):
        acc = (acc.astype(np.float64) + np.outer(a[:, k].astype(np.float64), b[k].astype(np.float64))).astype(np.float32)
    return acc


# The 256x256 tile, the 64x128 and the 128x128 one, and the latter in K slices.
SHAPES = [(4096, 64, 4096), (4096, 512, 4096), (1000, 64, 1000), (2200, 64, 2200), (1000, 512, 1000)]


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("share", [1.0, 0.35, 0.1, 0.02])
@pytest.mark.parametrize("right", [False, True])
def test_error_with_many_zeros_is_below_fp32_multiply_adds(m, k, n, share, right):
    rng = np.random.default_rng(m + k + int(100 * share) + right)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    x = b if right else a
    x *= rng.random(x.shape) < share
    got = U.matmul(a.ravel(), (m, k), (k, 1), 0, b.ravel(), (k, n), (n, 1), 0)
    rows, cols = slice(m - 200, m), slice(n - 200, n)
    want = a[rows].astype(np.float64) @ b[:, cols].astype(np.float64)
    err = lambda v: np.linalg.norm(v.astype(np.float64) - want) / np.linalg.norm(want)
    assert err(got[rows, cols]) < err(_fma(a[rows], b[:, cols]))


@pytest.mark.parametrize("m,k,n", [(4096, 100, 4096), (2200, 300, 2200), (1000, 1000, 1000), (300, 784, 500)])
def test_equal_rows_and_columns_give_equal_bits(m, k, n):
    """One row (column) repeated: every row (column) of the result is the same."""
    rng = np.random.default_rng(m + k)
    row, b = rng.standard_normal(k).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    got = U.matmul(row, (m, k), (0, 1), 0, b.ravel(), (k, n), (n, 1), 0)
    assert np.array_equal(got, np.broadcast_to(got[0], got.shape))
    a, col = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    got = U.matmul(a.ravel(), (m, k), (k, 1), 0, np.repeat(col, n), (k, n), (n, 1), 0)
    assert np.array_equal(got, np.broadcast_to(got[:, :1], got.shape))


@pytest.mark.parametrize("m,n", [(4096, 4096), (1000, 1000), (64, 200)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
def test_outer_products_are_correctly_rounded(m, n, ta, tb):
    """K = 1, where an operand's only column may be read as either layout."""
    rng = np.random.default_rng(m + n)
    a, b = rng.standard_normal((m, 1)).astype(np.float32), rng.standard_normal((1, n)).astype(np.float32)
    got = U.matmul(a.ravel(), (m, 1), (1, m) if ta else (1, 1), 0, b.ravel(), (1, n), (1, 1) if tb else (n, 1), 0)
    assert np.array_equal(got, a * b)
