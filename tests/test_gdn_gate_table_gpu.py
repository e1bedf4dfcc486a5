"""A prompt chunk's gated rows straight into the output projection's wide table (gdn_prefill_gate_table), against the rows by
themselves and the table made of them: the same bytes."""
import ctypes

import numpy as np
import pytest

import splash_amd
from tests import oracle as orc
from tests.test_wide_kernels_gpu import TableParams, table_bytes, wide_tiles

pytestmark = pytest.mark.gpu

TILED, SIGMOID, FLOAT_NORM = 1, 2, 4


class PrefillParams(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in ("key_heads", "value_heads", "conv_dim", "packed_width", "flags", "layer", "tokens", "first")] + \
               [(n, ctypes.c_uint64) for n in ("conv_layer_bytes", "recurrent_layer_bytes", "convolution_state_bytes", "current_cell", "next_cell")]


assert ctypes.sizeof(PrefillParams) == 72


# one super-block and the widest row; heads that end inside a wave's turn; rows that end inside a tile and at one's end
@pytest.mark.parametrize("key_heads,value_heads,tokens,flags", [(1, 2, 1, 0), (2, 6, 61, TILED), (9, 18, 128, SIGMOID), (16, 32, 130, TILED | FLOAT_NORM),
                                                                (16, 64, 17, 0)])
def test_gated_rows_as_a_table_are_the_table_of_the_rows(backend, key_heads, value_heads, tokens, flags):
    print(f"case gdn gate table {key_heads}/{value_heads} tokens={tokens} flags={flags}", flush=True)
    rng = np.random.default_rng(value_heads)
    width, conv, tiles = value_heads * 128, (2 * key_heads + value_heads) * 128, wide_tiles(tokens)
    packed_width = conv + width + 2 * value_heads
    recurrent = rng.standard_normal((tokens, width)).astype(np.float32)
    recurrent[tokens // 2] = 0
    recurrent[-1, 5], recurrent[0, 7] = np.inf, np.nan
    rows = backend.from_array(orc.f32_to_bf16(recurrent))
    packed = backend.from_array(orc.f32_to_bf16(rng.standard_normal((tokens, packed_width)).astype(np.float32) * 3))
    norm = (1 + 0.1 * rng.standard_normal(128)).astype(np.float32)
    weight = backend.from_array(norm if flags & FLOAT_NORM else orc.f32_to_bf16(norm))
    p = PrefillParams(key_heads, value_heads, conv, packed_width, flags, 0, tokens, 0)
    hidden = backend.allocate_buffer(tokens * width * 2)
    want, got = backend.allocate_buffer(table_bytes(width, tiles)), backend.allocate_buffer(table_bytes(width, tiles))
    want.fill(0xA5)
    got.fill(0xA5)
    grid = (64 * -(-16 * tiles // 64), 1, 1)
    graph = splash_amd.CommandGraph()
    graph.add("gdn_prefill_gate", [rows, packed, weight, hidden], p, (value_heads, -(-tokens // 16), 1))
    graph.add("gguf_wide_table", [hidden, hidden, want], TableParams(width, tokens, tiles, 0), grid)
    graph.add("gdn_prefill_gate_table", [rows, packed, weight, got], p, grid)
    backend.run(graph)
    assert np.array_equal(got.download(), want.download())
