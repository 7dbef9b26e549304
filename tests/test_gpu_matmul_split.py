"""The matmul tiles' three-piece bf16 split (gemm_tile.h) where it could go wrong.

Every float is the exact sum of three bf16 pieces, so a product with a signed
permutation matrix must return the operand's own floats bit for bit, whatever
their exponents: each output is one value times +-1 plus zeros, and every
addition of it is exact.  Values the pieces cannot hold (below 2^-110 with low
bits set, infinities, NaN, floats above bf16's largest) take the fp32 tile,
whose results have to be those of IEEE arithmetic.
"""
import numpy as np
import pytest

import gpu_util as U
import oracle as O

pytestmark = pytest.mark.gpu


def _stored(x, transposed):
    """x as the matmul takes it: plain rows, or its transpose's storage."""
    r, c = x.shape
    return (np.ascontiguousarray(x.T).ravel(), ((r, c), (1, r), 0)) if transposed else (x.ravel(), ((r, c), (c, 1), 0))


def _product(a, b, ta, tb):
    sa, la = _stored(a, ta)
    sb, lb = _stored(b, tb)
    return U.matmul(sa, *la, sb, *lb).reshape(a.shape[0], b.shape[1])


def _permutation(rng, n):
    """(P, column of each row, signs): x @ P moves column k of x to perm[k], times sign[k]."""
    perm, sign = rng.permutation(n), rng.choice(np.array([-1.0, 1.0], np.float32), n)
    p = np.zeros((n, n), np.float32)
    p[np.arange(n), perm] = sign
    return p, perm, sign


def _moved(x, perm, sign):
    want = np.empty_like(x)
    want[:, perm] = x * sign
    return want


def _floats(rng, shape, lo, hi):
    """Floats of random sign and mantissa and an exponent field of lo..hi."""
    bits = rng.integers(0, 1 << 23, shape, dtype=np.uint32)
    bits |= rng.integers(lo, hi + 1, shape, dtype=np.uint32) << np.uint32(23)
    bits |= rng.integers(0, 2, shape, dtype=np.uint32) << np.uint32(31)
    return bits.view(np.float32)


# One shape a kernel: the 256x256 tile (whole and ragged), stream-K on it, the
# 128x128 tile over split K (ragged), the 64x128 tile, and K of one partial
# slot, whole slots and one more.
SHAPES = [(4096, 4096), (4095, 4093), (3072, 3072), (1000, 1000), (64, 4096), (70, 33), (70, 40), (500, 48), (500, 65)]
LAYOUTS = [(False, False), (True, False), (False, True), (True, True)]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_every_bit_of_a_float_comes_through(m, n, ta, tb):
    rng = np.random.default_rng(m + 3 * n + 5 * ta + 7 * tb)
    p, perm, sign = _permutation(rng, n)
    # exponents from 2^-103 (the lowest bit at bf16's smallest subnormal, 2^-126 - 7) up to 2^126
    x = _floats(rng, (m, n), 24, 253)
    assert np.array_equal(_product(x, p, ta, tb) + 0.0, _moved(x, perm, sign) + 0.0)
    # the other operand: rows moved
    y = _floats(rng, (n, max(m, 33)), 24, 253)
    got = _product(p, y, ta, tb) if n > 32 else None
    if got is not None:
        assert np.array_equal(got + 0.0, y[perm] * sign[:, None] + 0.0)


@pytest.mark.parametrize("m,n", [(4096, 4096), (3072, 3072), (1000, 1000), (64, 4096), (70, 40)])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_values_the_pieces_cannot_hold(m, n, ta, tb):
    """A few floats out of the split's range: tiny ones (their low bits below
    bf16's smallest subnormal, subnormal floats among them) and floats that
    round to infinity in bf16 come through bit for bit; an infinity and a NaN
    give exactly the outputs 0 * x gives."""
    rng = np.random.default_rng(2 * m + n + ta + 2 * tb)
    p, perm, sign = _permutation(rng, n)
    x = _floats(rng, (m, n), 100, 140)
    rows = rng.choice(m, 8, replace=False)
    cols = rng.integers(0, n, 8)
    x[rows[0], cols[0]] = np.float32(3.4e38)
    x[rows[1], cols[1]] = np.float32(1.2345678e-36)
    x[rows[2], cols[2]] = np.float32(-1.2345678e-35)
    x[rows[3], :] = _floats(rng, n, 1, 15)
    want = _moved(x, perm, sign)
    assert np.array_equal(_product(x, p, ta, tb) + 0.0, want + 0.0)
    x[rows[5], cols[5]] = np.inf
    x[rows[6], cols[6]] = -np.inf
    x[rows[7], cols[7]] = np.nan
    got = _product(x, p, ta, tb)
    for r, c in ((rows[5], cols[5]), (rows[6], cols[6])):
        want[r, :] = np.nan
        want[r, perm[c]] = x[r, c] * sign[c]
    want[rows[7], :] = np.nan
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = ~np.isnan(want)
    assert np.array_equal(got[fin] + 0.0, want[fin] + 0.0)


@pytest.mark.parametrize("k", [1, 7, 8, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 129])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_slot_edges_within_tolerance(k, ta, tb):
    """K around the slots' ends (partial slots, one to three slots, and on),
    normal inputs: every element within the matmul tolerance."""
    m, n = 100, 131
    rng = np.random.default_rng(k + 2 * ta + tb)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    got = _product(a, b, ta, tb)
    want = a.astype(np.float64) @ b.astype(np.float64)
    bound = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    # Six additions into the accumulator per slot of 16 k, each off by at most
    # an ulp (2^-23) of a sum no larger than the bound, and 2^-24 for the three
    # products left out.
    assert (np.abs(got - want) <= (12 * -(-k // 16) + 1) * 2.0 ** -24 * bound).all()
    ref = O.matmul_threads(a, b, threads=4).reshape(m, n)
    assert (np.abs(got.astype(np.float64) - ref) <= 1e-5 * np.sqrt(k) * bound).all()


@pytest.mark.parametrize("k", [64, 512, 4096])
@pytest.mark.parametrize("positive", [False, True])
def test_error_against_64_bits_is_below_sequential_fp32(k, positive):
    """The 2-norm error against float64 is below that of the reference's own
    sequential fp32 order on the same inputs."""
    m = n = 256
    rng = np.random.default_rng(k + positive)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    if positive:
        a, b = np.abs(a), np.abs(b)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err = lambda x: np.linalg.norm(x.astype(np.float64) - want) / np.linalg.norm(want)
    ref = O.matmul_threads(a, b, threads=4).reshape(m, n)
    assert err(_product(a, b, False, False)) < err(ref)


def test_stride_0_and_long_row_strides():
    """Operands with a zero row stride (an expanded row) and with rows far apart."""
    rng = np.random.default_rng(9)
    m, k, n = 130, 50, 70
    row = rng.integers(-4, 5, k).astype(np.float32)
    b = rng.integers(-4, 5, (k, n)).astype(np.float32)
    got = U.matmul(row, (m, k), (0, 1), 0, b.ravel(), (k, n), (n, 1), 0)
    assert np.array_equal(got.reshape(m, n), np.tile(row @ b, (m, 1)))
    far = np.zeros(m * 5003, np.float32)
    a = rng.integers(-4, 5, (m, k)).astype(np.float32)
    far.reshape(m, 5003)[:, 3:3 + k] = a
    got = U.matmul(far, (m, k), (5003, 1), 3, b.ravel(), (k, n), (n, 1), 0)
    assert np.array_equal(got.reshape(m, n), a @ b)


@pytest.mark.parametrize("m,k,n", [(4096, 100, 4096), (1000, 1000, 1000), (512, 4096, 4096), (70, 120, 200)])
@pytest.mark.parametrize("right", [False, True])
def test_sums_that_overflow(m, k, n, right):
    """Values whose pieces are finite, and whose sums reach float's largest.  v is
    the float below 2^127: 2 v is the largest float, and the leading pieces of
    two v (2^127 each) add up to infinity, which fp32 arithmetic does not.  On
    one tile, in K slices and in stream-K's pieces; the other operand is ones."""
    v = np.nextafter(np.float32(2.0 ** 127), np.float32(0))
    top, inf = np.finfo(np.float32).max, np.float32(np.inf)
    at = [3, 5, k // 2, k - 9, k - 1]  # a group of 8 k, others, the last one
    rows, want = [], []
    for i in range(5):
        for j in range(i):
            rows += [{at[i]: v, at[j]: v}, {at[i]: -v, at[j]: -v}]
            want += [top, -top]
    rows += [{p: v for p in at[:3]}, {p: v for p in at[2:]}, {p: -v for p in at[::2]}]
    want += [inf, inf, -inf]
    x = np.zeros((n if right else m, k), np.float32)
    expected = np.zeros(x.shape[0], np.float32)
    for i, (row, w) in enumerate(zip(rows, want)):
        x[7 + 2 * i, list(row)] = list(row.values())
        expected[7 + 2 * i] = w
    back = 7 + 2 * len(rows)
    x[back, at] = [v, v, -v, -v, v]  # 2 v on the way, v in the end, in whatever order
    expected[back] = v
    other = np.ones((k, m if right else n), np.float32)
    got = _product(other.T, x.T, False, False).T if right else _product(x, other, False, False)
    assert np.array_equal(got, np.broadcast_to(expected[:, None], got.shape))
