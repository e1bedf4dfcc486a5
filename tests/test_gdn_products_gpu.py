"""The products of a verify block's rows with the committed state, which all rows of a block share on the matrix cores."""
import numpy as np
import pytest

from tests import oracle as orc
from tests.gdn_case import make_rows, make_state, make_tree
from tests.test_gdn_gpu import Chunk, Layer

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


def _half_wave_products(state, z):
    """What the products were before they ran on the matrix cores: fp32 sums of four columns a lane in column order, the 32
    lanes' as a tree."""
    terms = state.astype(np.float32) * z.astype(np.float32)
    terms = terms.reshape(*terms.shape[:-1], 32, 4)
    sums = np.zeros(terms.shape[:-1], np.float32)
    for i in range(4):
        sums = sums + terms[..., i]
    while sums.shape[-1] > 1:
        sums = sums[..., 0::2] + sums[..., 1::2]
    return sums[..., 0]


def test_the_products_lose_no_precision(backend):
    """The sums' error against 64 bits, of states that are orthogonal to the block's queries: the terms cancel, and what
    leaves in bf16 is the sums' own error and the states' rounding. No gate takes part: betas of 0, decays of 1, values of 0, and
    outputs that lie far below the norm's epsilon, which makes it a factor."""
    rng = np.random.default_rng(31)
    layer = Layer(backend, rng, 16, 32, lanes=1, float_norm=True, cells=4)
    shape, rows = layer.shape, 16
    vw, kw = shape.value_heads * 128, shape.key_heads * 128
    conv_w = layer.conv_w.copy()
    conv_w[2 * kw:] = 0                                                # values of zero
    layer.weights["convolution_weights"] = backend.from_array(conv_w)
    gate = 8.0
    packed = orc.bf16_to_f32(make_rows(rng, shape, rows))
    packed[:, shape.conv_dim:shape.conv_dim + vw] = gate
    packed[:, shape.conv_dim + vw:] = -400.0                           # sigmoid 0, softplus 0
    packed = orc.f32_to_bf16(packed)
    conv, state = make_state(rng, shape)
    layer.write_cell(0, 0, conv, state)
    run = Chunk(layer, rows).run(packed, 0, 0, 1)
    assert not run["beta"].any() and (run["decay"] == 1).all() and not run["values"].any()
    queries = orc.bf16_to_f32(run["queries"]).reshape(rows, shape.key_heads, 128).astype(np.float64)
    queries = np.repeat(queries, shape.value_heads // shape.key_heads, axis=1).transpose(1, 0, 2)      # [head][row][column]
    wide = state.astype(np.float64)
    state = (wide - wide @ np.linalg.pinv(queries) @ queries).astype(np.float32)
    layer.write_cell(0, 0, conv, state)
    (hidden,) = layer.step([(0, packed, 0, 0, 0, 2)])
    got = orc.bf16_to_f32(hidden).reshape(rows, shape.value_heads, 128).transpose(1, 0, 2).astype(np.float64)   # [head][row][value]
    got /= layer.norm.astype(np.float64) * (gate / (1 + np.exp(-gate))) * 1e3
    exact = queries @ state.astype(np.float64).transpose(0, 2, 1)
    norm = np.sqrt((queries ** 2) @ (state.astype(np.float64) ** 2).transpose(0, 2, 1))
    error = lambda x: float(np.sqrt((((x - exact) / norm) ** 2).mean()))
    before = error(_half_wave_products(state[:, None], queries[:, :, None]).astype(np.float64))
    print(f"case gdn products error {error(got):.3g} of the terms' norm (half-wave tree {before:.3g}, residue {error(0 * exact):.3g})", flush=True)
    # 65536 sums: the two means scatter by 0.3 %; the outputs' three roundings to bf16 add 1 % of the outputs
    assert error(got) <= 1.02 * before
