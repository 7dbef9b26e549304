"""How the pointwise kernels reach memory (trs_pointwise_plan_access, no device):
which of the launches of tests/test_gpu_pointwise_ragged.py run on vectors at any
float, which transpose through LDS, and which stay scalar."""
import pytest

from test_gpu_pointwise_ragged import THROUGH_LDS, XPOSE
from trs_backend import abi
from trs_backend.abi import layout_of

XPOSE_VARIANT = 3


def access(*layouts, out, **kw):
    return abi.pointwise_plan_access(list(layouts), out, **kw)


@pytest.mark.parametrize("cols", [2, 3, 4, 5, 63, 257, 1001])
@pytest.mark.parametrize("rows", [2, 37])
def test_rows_of_any_length_at_any_float_are_vectors_from_4_columns(rows, cols):
    x, b = layout_of((rows, cols)), layout_of((cols,))
    assert access(x, b, out=x) == (cols >= 4, False)
    base = [0x20000000000 + 4 * rows * cols, 0x30000000000]  # base[1] of a batch of two
    assert access(x, b, out=x, bases=base) == (cols >= 4, False)
    assert abi.pointwise_plan([x, b], x).vec == (cols >= 4 and cols % 4 == 0)  # aligned ones


@pytest.mark.parametrize("cols", [64, 66, 67, 256, 259])
def test_byte_operands_are_vectors_on_whole_quads(cols):
    x, b = layout_of((41, cols)), layout_of((cols,))
    assert access(x, b, x, out=x, elem_bytes=[4, 4, 1]) == (cols % 4 == 0, False)


@pytest.mark.parametrize("nb,t,x", XPOSE + THROUGH_LDS)
def test_transposed_operands_vector_and_lds(nb, t, x):
    a, b, c = layout_of((nb, 1, x)), layout_of((1, t, x)), layout_of((nb, t, x), (t * x, 1, t))
    out = layout_of((nb, t, x))
    plan = abi.pointwise_plan([a, b, c], out, roles=True)
    assert plan.variant == XPOSE_VARIANT
    # rows off the 128-byte lines and 64 x 256 tiles (t by x) at least 0.55 full
    lds = (nb, t, x) in THROUGH_LDS
    for roles in (False, True):
        assert access(a, b, c, out=out, roles=roles) == (True, lds)
    # two transposed operands stay in registers
    assert access(c, c, b, out=out, roles=True) == (True, False)
