"""Pointwise launches whose rows are of any length and start at any float.

The rows and transposing kernels read and write whole float4 there, moved back
to end at the row's (or column's) edge, and the transposing one goes through
LDS where the output's rows are not whole lines apart.  add, mul and relu round
once per element, so every result equals numpy's float32 bit for bit.
"""
import ctypes

import numpy as np
import pytest

import gpu_util as U
from trs_backend import abi
from trs_backend.abi import check, layout_of

pytestmark = pytest.mark.gpu


def _bits(x):
    return np.ascontiguousarray(x, np.float32).view(np.uint32)


def _same(got, want):
    assert got.shape == want.shape
    assert np.array_equal(_bits(got), _bits(want))


def _normal(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 6, 7, 63, 64, 65, 255, 256, 257, 258, 259, 1001, 1023, 1025])
@pytest.mark.parametrize("rows", [2, 37])
def test_rows_of_any_length(rows, cols):
    import torch_rs
    rng = np.random.default_rng(rows + cols)
    x, b = _normal(rng, 2, rows, cols), _normal(rng, cols)
    base = torch_rs.tensor(x, device="cuda")
    db = torch_rs.tensor(b, device="cuda")
    fused = torch_rs.fuse(lambda p, q: (p + q).relu())
    for i in range(2):  # base[1] starts rows * cols floats on: at any float
        want = x[i] + b
        _same((base[i] + db).numpy(), want)
        _same(fused(base[i], db).numpy(), np.where(want > 0, want, np.float32(0)))
        _same((base[i] * base[1 - i]).numpy(), x[i] * x[1 - i])


@pytest.mark.parametrize("cols", [5, 257, 1003])
def test_in_place_over_ragged_rows(cols):
    """The output is the first operand's own view: the lane that computes a
    row's last columns again must not read what another has written."""
    rng = np.random.default_rng(cols)
    rows = 300
    x, b = _normal(rng, rows, cols), _normal(rng, cols)
    dx, db = U.dev(x), U.dev(b)
    lx, lb = layout_of((rows, cols)), layout_of((cols,))
    check(abi.lib.trs_binary_f32(abi.TRS_ADD, dx.ptr, ctypes.byref(lx), db.ptr, ctypes.byref(lb), dx.ptr,
                                 ctypes.byref(lx)))
    _same(dx.to_numpy(count=rows * cols).reshape(rows, cols), x + b)


@pytest.mark.parametrize("cols", [64, 66, 67, 256, 259])
def test_byte_mask_over_ragged_rows(cols):
    import torch_rs
    rng = np.random.default_rng(cols)
    h, bias, mask = _normal(rng, 41, cols), _normal(rng, cols), (rng.random((41, cols)) < 0.5).astype(np.uint8)
    dh, db = torch_rs.tensor(h, device="cuda"), torch_rs.tensor(bias, device="cuda")
    dm = torch_rs.nn.functional.keep_mask(mask)
    act = torch_rs.fuse(lambda z, b, m: ((z + b).relu() * m) * 2.0)
    z = h + bias
    _same(act(dh, db, dm).numpy(), (np.where(z > 0, z, np.float32(0)) * mask) * np.float32(2.0))


# (batch, t, x): the transposing tiles' edges (128 x 64, and 64 x 256 through
# LDS), sizes under a float4, and rows that are whole lines apart.
XPOSE = [(1, 3, 5), (2, 4, 4), (2, 5, 7), (1, 31, 128), (1, 32, 127), (3, 32, 129), (2, 33, 255), (2, 63, 257),
         (2, 64, 256), (2, 65, 260), (1, 66, 511), (2, 67, 513), (2, 127, 65), (1, 129, 66), (2, 130, 1001),
         (1, 500, 259), (2, 131, 1024), (5, 40, 300)]


@pytest.mark.parametrize("nb,t,x", XPOSE)
def test_transposed_operand_at_every_edge(nb, t, x):
    import torch_rs
    rng = np.random.default_rng(nb + 3 * t + 7 * x)
    a, b, c, d = _normal(rng, nb, 1, x), _normal(rng, 1, t, x), _normal(rng, nb, x, t), _normal(rng, nb, x, t)
    da, db, dc, dd = (torch_rs.tensor(v, device="cuda") for v in (a, b, c, d))
    ct, dt = c.transpose(0, 2, 1), d.transpose(0, 2, 1)
    _same(torch_rs.fuse(lambda p, q, r: (p + q) * r)(da, db, dc.mT).numpy(), (a + b) * ct)
    _same(((da + db) * dc.mT).numpy(), (a + b) * ct)
    full = a + b  # contiguous, unit stride along x
    _same((torch_rs.tensor(full, device="cuda") + dc.mT).numpy(), full + ct)
    _same(torch_rs.fuse(lambda p, q, r: (p * q) + r)(dc.mT, dd.mT, db).numpy(), (ct * dt) + b)
    col = _normal(rng, nb, t, 1)  # constant along x
    _same(torch_rs.fuse(lambda p, q: p * q)(torch_rs.tensor(col, device="cuda"), dc.mT).numpy(), col * ct)


# Those that run on the tiles through LDS (64 t by 256 x, at least 0.55 full, and a
# batch of 4 or 8, which the direct tiles would walk): t and x around the tiles'
# edges, a last tile of one row or column, every residue mod 4, and the least full.
THROUGH_LDS = [(8, 36, 253), (4, 64, 144), (4, 64, 145), (4, 63, 146), (4, 63, 147), (4, 62, 255), (4, 64, 254),
               (4, 129, 1023), (4, 130, 1021), (8, 131, 1022), (4, 64, 769), (4, 64, 770), (4, 64, 771), (4, 127, 511),
               (4, 125, 700), (8, 128, 510), (4, 130, 1001)]


def _lds_operands(nb, t, x):
    rng = np.random.default_rng(nb + 3 * t + 7 * x)
    return _normal(rng, nb, 1, x), _normal(rng, 1, t, x), _normal(rng, nb, x, t), _normal(rng, nb, t, 1), _normal(rng, 1)


def _runs_through_lds(nb, t, x, roles=True):
    """(a + b) * c.mT fused, or c.mT and a whole operand eager."""
    whole, ct = layout_of((nb, t, x)), layout_of((nb, t, x), (t * x, 1, t))
    lays = [layout_of((nb, 1, x)), layout_of((1, t, x)), ct] if roles else [whole, ct]
    return abi.pointwise_plan_access(lays, whole, roles=roles) == (True, True)


@pytest.mark.parametrize("nb,t,x", THROUGH_LDS)
def test_lds_tiles_at_every_edge(nb, t, x):
    import torch_rs
    assert _runs_through_lds(nb, t, x)
    host = a, b, c, col, scalar = _lds_operands(nb, t, x)
    da, db, dc, dcol, ds = (torch_rs.tensor(v, device="cuda") for v in host)
    ct, full = c.transpose(0, 2, 1), a + b
    _same(torch_rs.fuse(lambda p, q, r: (p + q) * r)(da, db, dc.mT).numpy(), full * ct)
    # five inputs: the others are read after the barrier
    five = torch_rs.fuse(lambda p, q, r, u, v: ((p + q) * r - u) * v)
    _same(five(da, db, dc.mT, dcol, ds).numpy(), (full * ct - col) * scalar)


@pytest.mark.parametrize("nb,t,x", [(128, 61, 413), (256, 64, 255), (65, 80, 1021), (43, 130, 511), (257, 36, 254)])
def test_lds_tiles_eager(nb, t, x):
    """From a block per CU (256) on, whatever the batch."""
    import torch_rs
    assert _runs_through_lds(nb, t, x, roles=False)
    a, b, c, _, _ = _lds_operands(nb, t, x)
    full, ct = a + b, c.transpose(0, 2, 1)
    got = torch_rs.tensor(full, device="cuda") + torch_rs.tensor(c, device="cuda").mT
    _same(got.numpy(), full + ct)


def test_loop_over_lds_tiles_of_a_walked_batch():
    """Fewer blocks than tiles: each block takes several LDS tiles."""
    import torch_rs
    nb, t, x = 4, 150, 601
    assert _runs_through_lds(nb, t, x)
    a, b, c, _, _ = _lds_operands(nb, t, x)
    da, db, dc = (torch_rs.tensor(v, device="cuda") for v in (a, b, c))
    check(abi.lib.trs_debug_pointwise_grid_cap(3))
    try:
        _same(torch_rs.fuse(lambda p, q, r: (p + q) * r)(da, db, dc.mT).numpy(), (a + b) * c.transpose(0, 2, 1))
    finally:
        check(abi.lib.trs_debug_pointwise_grid_cap(0))


def test_transposed_views_at_any_float_and_higher_rank():
    import torch_rs
    rng = np.random.default_rng(4)
    base = _normal(rng, 3, 301, 71)
    other = _normal(rng, 71, 301)
    db, do = torch_rs.tensor(base, device="cuda"), torch_rs.tensor(other, device="cuda")
    for i in range(3):  # base[i] starts 301 * 71 * i floats on
        _same((do + db[i].mT).numpy(), other + base[i].T)
        _same(torch_rs.fuse(lambda p, q: (p + q) * q)(do, db[i].mT).numpy(), (other + base[i].T) * base[i].T)
    p = _normal(rng, 2, 3, 131, 45)
    q = _normal(rng, 2, 1, 45, 131)
    dp, dq = torch_rs.tensor(p, device="cuda"), torch_rs.tensor(q, device="cuda")
    _same((dq * dp.mT).numpy(), q * p.swapaxes(2, 3))


def test_transposing_loop_over_lds_tiles():
    """Fewer blocks than tiles: each block walks several LDS tiles."""
    import torch_rs
    rng = np.random.default_rng(6)
    a, c = _normal(rng, 3, 150, 601), _normal(rng, 3, 601, 150)
    da, dc = torch_rs.tensor(a, device="cuda"), torch_rs.tensor(c, device="cuda")
    check(abi.lib.trs_debug_pointwise_grid_cap(2))
    try:
        _same((da + dc.mT).numpy(), a + c.transpose(0, 2, 1))
        _same(torch_rs.fuse(lambda p, q: p * q + p)(da, dc.mT).numpy(), a * c.transpose(0, 2, 1) + a)
    finally:
        check(abi.lib.trs_debug_pointwise_grid_cap(0))
