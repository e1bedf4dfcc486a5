"""The experts' weighted sum of a prompt chunk's rows, eight columns a thread, against a column a thread."""
import ctypes

import numpy as np
import pytest

import splash_amd
from tests import oracle as orc

pytestmark = pytest.mark.gpu


class Combine(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in ("rows", "hidden", "top_k", "table_tiles")]


@pytest.mark.parametrize("rows,hidden,top_k", [(1, 8, 1), (3, 2056, 7), (5, 2048, 8), (2, 4104, 9), (17, 264, 17)])
def test_combined_rows_are_the_same_bits(backend, rows, hidden, top_k):
    """One vector a row, a second workgroup of one thread, as many routes as are loaded together and one more."""
    print(f"case moe combine rows={rows} hidden={hidden} top_k={top_k}", flush=True)
    rng = np.random.default_rng(rows)
    slots = rows * top_k
    bf16 = lambda *shape: backend.from_array(orc.f32_to_bf16(rng.standard_normal(shape).astype(np.float32)))
    experts, residual = bf16(slots, hidden), bf16(rows, hidden)
    route = backend.from_array(rng.permutation(slots).astype(np.uint32))
    weights = backend.from_array(rng.random(slots).astype(np.float32))
    wide, narrow = (backend.from_array(np.full(rows * hidden, 0xA5A5, np.uint16)) for _ in range(2))
    p = Combine(rows, hidden, top_k, 0)
    graph = splash_amd.CommandGraph()
    graph.add("moe_combine", [experts, route, weights, residual, narrow, narrow, narrow], p, (rows, (hidden + 255) // 256, 1), (256, 1, 1))
    graph.add("moe_combine_rows", [experts, route, weights, residual, wide], p, (rows, (hidden + 2047) // 2048, 1), (256, 1, 1))
    backend.run(graph)
    assert np.array_equal(wide.download(), narrow.download())
