"""Products whose operands hold values that the bf16 pieces cannot hold whole
(below 2^-110): the tile's own judgement of whether the lost bits can show.

Every output has to be within fp32 rounding of its own products, however small:
|error| <= (K + 2) * 2^-24 * (|A| @ |B|), and K / 2 of float's smallest
subnormal where that is more.
"""
import time

import numpy as np
import pytest

import gpu_util as U
from test_gpu_matmul import _layouts

pytestmark = pytest.mark.gpu


def _check(a, b, ta, tb):
    m, k = a.shape
    n = b.shape[1]
    sa, la, sb, lb = _layouts(a, b, ta, tb)
    got = U.matmul(sa, *la, sb, *lb).reshape(m, n)
    step = max(1, m // 300)  # float64 products of some rows, the last among them
    rows = np.unique(np.r_[0:m:step, m - 1])
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    bound = (k + 2) * 2.0 ** -24 * (np.abs(a[rows]).astype(np.float64) @ np.abs(b).astype(np.float64)) + k * 2.0 ** -150
    assert (np.abs(got[rows] - want) <= bound).all()


# The 256x256 tile, stream-K, 128x128 in slices, 64x128 unsplit and in slices.
SHAPES = [(4096, 100, 4096), (512, 4096, 4096), (1000, 1000, 1000), (70, 120, 200), (300, 784, 500)]


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
@pytest.mark.parametrize("right", [False, True])
@pytest.mark.parametrize("kind", ["some", "late", "row", "all", "zeros", "wide"])
def test_tiny_values(m, k, n, ta, tb, right, kind):
    rng = np.random.default_rng(m + k + 2 * ta + right)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    x = b.T if right else a  # rows of k values
    tiny = (rng.standard_normal(x.shape) * 2.0 ** -115).astype(np.float32)
    if kind == "some":  # among ordinary ones, from the first slots on
        x[:] = np.where(rng.random(x.shape) < 0.02, tiny, x)
    elif kind == "late":  # none in the first slots
        x[::7, k - 20] = tiny[::7, k - 20]
    elif kind == "row":  # a row of nothing else: its outputs are as small
        x[x.shape[0] - 2] = tiny[0]
        x[5, : k // 2] = tiny[5, : k // 2]
    elif kind == "all":
        x[:] = tiny
    elif kind == "zeros":  # rows of one tiny value and zeros, and of zeros
        x[1::3] = 0
        x[2::3] = 0
        x[2::3, k // 2] = tiny[2::3, 0]
    else:  # rows from subnormals to 2^40
        x *= np.exp2(np.linspace(-148, 40, x.shape[0])).astype(np.float64)[:, None].astype(np.float32)
    _check(a, b, ta, tb)


def test_a_few_tiny_values_do_not_take_the_fp32_path():
    """One value of 2^-119 in every 64 rows of a dense operand: every tile looks
    its operands over once more (1.4 times the time without them, measured), and
    none is computed again on fp32 MFMA (2.7 times)."""
    import ctypes
    from trs_backend import abi
    n = 4096
    rng = np.random.default_rng(0)
    a, b = rng.standard_normal((n, n)).astype(np.float32), rng.standard_normal((n, n)).astype(np.float32)
    lay, db, out = abi.layout_of((n, n)), U.dev(b), U.out_buffer(n * n)

    def best(x):
        dx, times = U.dev(x), []
        for _ in range(8):
            abi.check(abi.lib.trs_synchronize())
            t = time.perf_counter()
            for _ in range(4):
                abi.check(abi.lib.trs_matmul_f32(dx.ptr, ctypes.byref(lay), db.ptr, ctypes.byref(lay), out.ptr,
                                                 ctypes.byref(lay)))
            abi.check(abi.lib.trs_synchronize())
            times.append(time.perf_counter() - t)
        return min(times)

    plain = best(a)
    a[::64, ::997] = 1.2345678e-36
    assert best(a) < 2 * plain
