"""The draft attention's merged rows as the activation table of the projection that reads them."""
import ctypes

import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc
from tests.test_draft_attention_gpu import D, KVH, RING, ROWS, WINDOW, bits

pytestmark = pytest.mark.gpu


class Merge(ctypes.Structure):
    _fields_ = [("lanes", ctypes.c_uint32), ("table_tiles", ctypes.c_uint32)]


@pytest.mark.parametrize("lanes", [1, 2, 3, 8])
def test_the_merge_leaves_the_table_pass_table(backend, lanes):
    """A row tile half empty, full, one over and the most lanes: the rows are those of the merge without a table, the table
    the one gguf_prepare_table makes of them."""
    print(f"case draft merge table lanes={lanes}", flush=True)
    rng = np.random.default_rng(lanes)
    op = ops.DraftAttention(5120, lanes)
    unit = lambda *shape: bits(rng.uniform(-1, 1, shape))
    rings = backend.from_array(unit(lanes * RING))
    grouped = backend.allocate_buffer(op.grouped_queries_bytes)
    grouped.upload(unit(lanes, KVH, 32, D))
    graph = splash_amd.CommandGraph()
    op.add_decode(graph, grouped, rings, [lane * 2 * RING for lane in range(lanes)], [(lane * 2 + 1) * RING for lane in range(lanes)],
                  backend.from_array(unit(lanes, KVH, ROWS, D)), backend.from_array(unit(lanes, KVH, D, ROWS)), [100 * lane for lane in range(lanes)])
    backend.run(graph)
    query_bytes = lanes * ROWS * 4096 * 2
    partials = grouped.view(query_bytes, op.grouped_queries_bytes - query_bytes)
    out, table = backend.allocate_buffer(query_bytes), backend.allocate_buffer(ops.gguf_table_bytes(4096, lanes * ROWS))
    graph = splash_amd.CommandGraph()
    graph.add("draft_attention_merge", [partials, out, table], Merge(lanes, (lanes * ROWS + 15) // 16), (KVH, lanes, 1), (1024, 1, 1))
    backend.run(graph)
    rows = out.download(np.uint16).reshape(lanes * ROWS, 4096)
    assert np.array_equal(rows.ravel(), grouped.download(np.uint16)[:rows.size])
    orc.assert_table_holds(table.download(np.uint8), rows, lambda count: ops.gguf_table_bytes(4096, count))
