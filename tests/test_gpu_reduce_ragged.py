"""Broadcast gradients over rows of any length, at any float: the staged
reduction's edge quads of chains, short chains and partial stages.  Every chain
is added in the reference's order from +0.0, so results equal a sequential
float32 sum bit for bit.
"""
import ctypes
import time

import numpy as np
import pytest

import gpu_util as U
from trs_backend import abi
from trs_backend.abi import check, layout_of

pytestmark = pytest.mark.gpu


def _same(got, want):
    assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))


def _normal(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("rows,cols", [(16, 4), (16, 5), (63, 64), (64, 15), (64, 17), (255, 33), (256, 1001),
                                       (300, 7), (511, 31), (513, 47), (1000, 1000), (2049, 10), (2050, 70000)])
def test_broadcast_gradients_of_any_width(rows, cols):
    """The add VJP over rows of any length: every chain added in the
    reference's order from +0.0 (numpy's float32 add.accumulate)."""
    rng = np.random.default_rng(rows + cols)
    up = _normal(rng, rows, cols)
    du, do = U.dev(up), U.out_buffer(cols)
    check(abi.lib.trs_reduce_to_shape_f32(du.ptr, ctypes.byref(layout_of((rows, cols))),
                                          ctypes.byref(layout_of((cols,))), do.ptr))
    want = np.zeros(cols, np.float32)
    for r in range(rows):
        want += up[r]
    _same(do.to_numpy(count=cols), want)


@pytest.mark.parametrize("kind", ["plain", "transposed", "row", "scalar"])
@pytest.mark.parametrize("nb,rows,cols", [(1, 300, 37), (3, 260, 50), (2, 64, 33), (1, 1028, 7)])
def test_broadcast_mul_gradients_of_any_width(nb, rows, cols, kind):
    rng = np.random.default_rng(nb + rows + cols)
    up = _normal(rng, nb, rows, cols)
    if kind == "transposed":
        store = _normal(rng, nb, cols, rows)
        other, st = store.transpose(0, 2, 1), (rows * cols, 1, rows)
    elif kind == "row":
        store = _normal(rng, cols)
        other, st = np.broadcast_to(store, (nb, rows, cols)), None
    else:
        store = _normal(rng, nb, rows, cols)
        other, st = store, (rows * cols, cols, 1)
    lo = layout_of((cols,)) if st is None else layout_of((nb, rows, cols), st)
    if kind == "scalar":  # every second column of wider rows: no vector along either dim
        store = _normal(rng, nb, rows, 2 * cols)
        other, lo = store[:, :, ::2], layout_of((nb, rows, cols), (rows * 2 * cols, 2 * cols, 2))
    du, dt, do = U.dev(up), U.dev(store), U.out_buffer(nb * cols)
    check(abi.lib.trs_mul_backward_f32(du.ptr, ctypes.byref(layout_of((nb, rows, cols))), dt.ptr, ctypes.byref(lo),
                                       ctypes.byref(layout_of((nb, 1, cols))), do.ptr))
    prod = up * other
    want = np.zeros((nb, cols), np.float32)
    for r in range(rows):
        want += prod[:, r]
    _same(do.to_numpy(count=nb * cols).reshape(nb, cols), want)


# Many outer kept indices of a few columns each, on both sides of the number of
# blocks (one per outer index and 32 columns, whole or not) up to which the staged
# kernel is taken on a 256-CU device: 1, 2, 4, 7 and 14 per CU.
@pytest.mark.parametrize("ko,rows,ki", [(256, 20, 4), (257, 20, 4), (256, 65, 33), (257, 65, 33), (1024, 130, 8),
                                        (1025, 130, 8), (1792, 260, 5), (1793, 260, 5), (3584, 513, 4), (3585, 513, 4),
                                        (1792, 513, 40), (1793, 513, 40)])
def test_broadcast_gradients_of_many_narrow_groups(ko, rows, ki):
    rng = np.random.default_rng(ko + rows + ki)
    up = _normal(rng, ko, rows, ki)
    du, do = U.dev(up), U.out_buffer(ko * ki)
    check(abi.lib.trs_reduce_to_shape_f32(du.ptr, ctypes.byref(layout_of((ko, rows, ki))),
                                          ctypes.byref(layout_of((ko, 1, ki))), do.ptr))
    want = np.zeros((ko, ki), np.float32)
    for r in range(rows):
        want += up[:, r]
    _same(do.to_numpy(count=ko * ki).reshape(ko, ki), want)


def test_narrow_groups_take_no_longer_than_twice_one_wide_one():
    """The same chains as 28,000 groups of 4 and as one of 112,000: 140 and about
    90 us (492 where 28,000 staged blocks each add 4 chains)."""
    up, out = U.out_buffer(112000 * 1000, 1.0), U.out_buffer(112000)

    def best(shape, kept):
        lu, ls, times = layout_of(shape), layout_of(kept), []
        for _ in range(8):
            check(abi.lib.trs_synchronize())
            t = time.perf_counter()
            for _ in range(10):
                check(abi.lib.trs_reduce_to_shape_f32(up.ptr, ctypes.byref(lu), ctypes.byref(ls), out.ptr))
            check(abi.lib.trs_synchronize())
            times.append(time.perf_counter() - t)
        return min(times)

    assert best((28000, 1000, 4), (28000, 1, 4)) < 2.5 * best((1000, 112000), (112000,))
