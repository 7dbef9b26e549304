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
    assert abi.pointwise_plan([a, b, c], out, roles=True).variant == XPOSE_VARIANT
    assert access(a, b, c, out=out, roles=True) == (True, (nb, t, x) in THROUGH_LDS)
    # without roles nothing is walked, and these are few blocks
    assert access(a, b, c, out=out) == (True, False)
    # two transposed operands stay in registers
    assert access(c, c, b, out=out, roles=True) == (True, False)


# 64 x 256 tiles (t by x): from a block per CU on, or where the direct tiles would
# walk 4 or 8 tuples of a batch; 0.55 full or more, and rows off the 128-byte lines.
@pytest.mark.parametrize("nb,t,x,lds", [(255, 64, 250, False), (256, 64, 250, True), (255, 64, 256, False),
                                        (9, 448, 703, False), (12, 448, 703, True), (22, 256, 748, True),
                                        (58, 528, 111, False), (512, 64, 140, False), (512, 64, 141, True),
                                        (6, 709, 420, False), (10, 709, 420, False), (8, 709, 420, True)])
def test_when_a_transposed_operand_goes_through_lds(nb, t, x, lds):
    a, b, c = layout_of((nb, 1, x)), layout_of((1, t, x)), layout_of((nb, t, x), (t * x, 1, t))
    assert access(a, b, c, out=layout_of((nb, t, x)), roles=True) == (True, lds)


@pytest.mark.parametrize("nb,t,x,lds", [(159, 64, 250, False), (160, 64, 250, True), (8, 448, 385, False),
                                        (43, 64, 933, True), (1, 1000, 777, False), (1, 3000, 3001, True)])
@pytest.mark.parametrize("roles", [False, True])
def test_with_a_second_whole_operand_through_lds_from_fewer_blocks(nb, t, x, lds, roles):
    y, c = layout_of((nb, t, x)), layout_of((nb, t, x), (t * x, 1, t))
    assert access(y, c, out=y, roles=roles) == (True, lds)


@pytest.mark.parametrize("cols,lanes", [(7843, 256), (1001, 256), (998, 256), (871, 256), (870, 64), (515, 64), (511, 64),
                                        (131, 64), (37, 64), (3679, 256), (1025, 64), (1400, 64)])
def test_ragged_rows_take_the_widest_blocks_where_they_fill_them(cols, lanes):
    """Rows off 16 bytes; aligned ones keep the block for the bytes it moves."""
    x, b = layout_of((300, cols)), layout_of((cols,))
    base = [0x20000000004, 0x30000000000]
    assert abi.pointwise_plan([x, b], x, bases=base).block == lanes
    aligned = layout_of((300, 4096))
    assert abi.pointwise_plan([aligned, layout_of((4096,))], aligned).block == 64
