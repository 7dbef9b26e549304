"""Products of few tiles: the 64x128 tile at shapes it does not divide, and its short K slices.

Small integers, whose products and sums are exact in any order, so the result
equals the float64 product bit for bit.
"""
import numpy as np
import pytest

import gpu_util as U
from test_gpu_matmul import _cu_count, _layouts, _matmul_without_allocations, _plan

pytestmark = pytest.mark.gpu

# (M, K, N) and the (tile_m, tile_n, splits) of a 256-CU device: one tile, K
# just below and at the least that splits, a ragged last slice, the most
# slices, the most tiles that split and one more, and the most unsplit tiles.
FEW = [((64, 64, 64), (64, 128, 1)), ((65, 127, 129), (64, 128, 1)), ((500, 128, 100), (64, 128, 2)),
       ((200, 400, 300), (64, 128, 7)), ((300, 784, 500), (64, 128, 10)), ((96, 6144, 96), (64, 128, 16)),
       ((1000, 1000, 500), (64, 128, 4)), ((1001, 997, 513), (128, 128, 7)), ((4095, 127, 500), (64, 128, 1)),
       ((4097, 127, 500), (128, 128, 1))]


def _ints(rng, shape):
    return rng.integers(-3, 4, shape).astype(np.float32)


@pytest.mark.parametrize("mkn,plan", FEW)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_few_tiles_exact_on_small_integers(mkn, plan, ta, tb):
    m, k, n = mkn
    if _cu_count() != 256:
        pytest.skip("plan expectations are those of a 256-CU device")
    got = _plan(m, k, n, ta, tb)
    assert (got[0], got[1], got[3]) == plan, got
    rng = np.random.default_rng(m + k + n)
    a, b = _ints(rng, (m, k)), _ints(rng, (k, n))
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    sa, la, sb, lb = _layouts(a, b, ta, tb)
    assert np.array_equal(U.matmul(sa, *la, sb, *lb).reshape(m, n), want)
    assert np.array_equal(_matmul_without_allocations(sa, *la, sb, *lb).reshape(m, n), want)


@pytest.mark.parametrize("nb,m,k,n", [(3, 100, 37, 70), (16, 300, 300, 300), (17, 300, 300, 300)])
def test_few_tiles_batched_exact_on_small_integers(nb, m, k, n):
    rng = np.random.default_rng(nb + m + k + n)
    a, b = _ints(rng, (nb, m, k)), _ints(rng, (nb, k, n))
    want = np.matmul(a.astype(np.float64), b.astype(np.float64)).astype(np.float32)
    got = U.matmul(a.ravel(), (nb, m, k), (m * k, k, 1), 0, b.ravel(), (nb, k, n), (k * n, n, 1), 0)
    assert np.array_equal(got.reshape(nb, m, n), want)
