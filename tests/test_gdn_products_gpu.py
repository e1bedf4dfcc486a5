"""The products of a verify block's rows with the committed state, which all rows of a block share on the matrix cores."""
import numpy as np
import pytest

from tests import oracle as orc
from tests.gdn_case import make_rows, make_state, make_tree
from tests.test_gdn_gpu import Layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 15, 16])
def test_a_row_depends_on_its_path_alone(backend, rows):
    """A tree block of 1 to 16 rows after a pending path: each row's output is, bit for bit, the output of the block that
    holds its path and no other row (every sum's order is the row's own), and a row whose values are not finite reaches
    only the rows below it."""
    print(f"case gdn products rows={rows}", flush=True)
    rng = np.random.default_rng(rows)
    layer = Layer(backend, rng, 2, 4, lanes=1, float_norm=True, cells=4)
    cell, pending = make_state(rng, layer.shape), make_rows(rng, layer.shape, 5)
    block, masks = make_rows(rng, layer.shape, rows), make_tree(rng, rows)
    layer.write_cell(0, 0, *cell)
    layer.step([(0, pending, 0, 0, 0, 1)])
    (whole,) = layer.step([(0, block, 0b11111, 1, 1, 2, masks)])
    assert np.isfinite(orc.bf16_to_f32(whole)).all()
    for row in {0, rows // 2, rows - 1}:
        path = [r for r in range(rows) if (masks[row] >> r) & 1]
        (alone,) = layer.step([(0, block[path], 0b11111, 1, 1, 3, [(2 << i) - 1 for i in range(len(path))])])
        assert np.array_equal(alone[-1], whole[row]), row
    if rows > 1:
        broken = block.copy()
        broken[rows // 2] = 0x7FC0   # NaN in every column
        (got,) = layer.step([(0, broken, 0b11111, 1, 1, 3, masks)])
        for row in range(rows):
            below = (masks[row] >> (rows // 2)) & 1
            assert below or np.array_equal(got[row], whole[row]), row
