"""The experts' gate/up pair of a prompt chunk from the rows' own tables, gathered (kernels/gguf_wide.hip), against the same
pair from a table of the slots: the same operands and the same sums, so the same bits."""
import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc
from tests.test_wide_kernels_gpu import FORMATS, TableParams, WideMoeParams, add_table, expected_places, place, table_bytes, wide_tiles

pytestmark = pytest.mark.gpu


def row_bytes(K):
    return -(-(K * 2 + K // 4) // 128) * 128


def rows_of_table(table, K, rows):
    """The rows' tables a wide table's bytes come to, without what fills their last lines."""
    values = table[:wide_tiles(rows) * K // 256 * 9216].reshape(-1, K // 256, 9, 4, 16, 16)
    values = values.transpose(0, 4, 1, 2, 3, 5).reshape(-1, K // 256, 9, 64)[:rows]
    return np.concatenate([values[:, :, :8].reshape(rows, -1), values[:, :, 8].reshape(rows, -1)], axis=1)


# tasks of every height up to T; a row of whole lines and rows whose lines are filled up; columns that end inside a group
@pytest.mark.parametrize("T,K", [(2, 256), (4, 768), (5, 512), (8, 512), (8, 2048)])
@pytest.mark.parametrize("name", list(FORMATS))
def test_gathered_rows_give_the_slots_bits(backend, name, T, K):
    fmt, N, experts, top_k, rows = FORMATS[name], 272, T + 2, 3, 700
    print(f"case wide gathered {name} T={T} K={K}", flush=True)
    rng = np.random.default_rng(T * K)
    routes = rows * top_k
    counts = [16 * height - int(rng.integers(0, 16)) for height in range(1, T + 1)] + [0]
    selected = rng.permutation(np.repeat(np.arange(experts), counts + [routes - sum(counts)]))
    b = place(backend, selected, experts, top_k, T)
    tiles = routes // 16 + experts
    images = [backend.from_array(np.concatenate([ops.pack_gguf_image(fmt, orc.make_native(fmt, N, K, seed + e), N, K) for e in range(experts)]))
              for seed in (1, 50)]
    x = backend.from_array(orc.f32_to_bf16((rng.standard_normal((rows, K)) * 0.02).astype(np.float32)))
    p = WideMoeParams()
    p.wide.input_size, p.wide.rows, p.wide.tiles, p.wide.out_stride, p.expert_bytes = K, rows, tiles, N, images[0].size_bytes // experts
    p.wide.cols[0], p.wide.groups = N, -(-N // 64)
    grid = (8 * -(-(tiles // T + experts) * p.wide.groups // 8), 1, 1)
    got = []
    for kind in ("slots", "rows"):
        out = backend.allocate_buffer(16 * tiles * N * 2)
        out.fill(0xA5)
        graph = splash_amd.CommandGraph()
        if kind == "slots":
            table = backend.allocate_buffer(table_bytes(K, tiles))
            table.fill(0xA5)
            graph.add("gguf_wide_moe_gather", [x, b["slot_row"], b["totals"], table], TableParams(K, rows, tiles, 0), (64 * -(-16 * tiles // 64), 1, 1))
            graph.add(f"gguf_wide_moe_{name}_t{T}_g", [images[0], images[1], table, out, b["tasks"], b["totals"]], p, grid)
        else:
            table = backend.allocate_buffer(rows * (row_bytes(K) + 4))
            table.fill(0xA5)
            graph.add("gguf_wide_rows", [x, table], TableParams(K, rows, tiles, 0), (rows, 1, 1))
            graph.add(f"gguf_wide_moe_{name}_t{T}_x", [images[0], images[1], table, out, b["tasks"], b["totals"], b["slot_row"]], p, grid)
        backend.run(graph)
        got.append(out.download(np.uint16))
    assert np.array_equal(got[0], got[1]) and (got[0] != 0xA5A5).any()


@pytest.mark.parametrize("rows,K", [(1, 256), (17, 1792), (130, 8192)])
def test_rows_tables_hold_what_the_wide_table_does(backend, rows, K):
    """The rows' tables of rows and of their norms, and the wide table written beside the latter."""
    print(f"case rows' tables {rows} K={K}", flush=True)
    rng = np.random.default_rng(rows)
    x = orc.f32_to_bf16((rng.standard_normal((rows, K)) * 10.0 ** rng.integers(-6, 7, (1, K))).astype(np.float32))
    x[0, 3], x[rows - 1, 0], x[rows // 2, :5] = 0x7F80, 0x7FC1, 0
    weight, tiles, size = orc.f32_to_bf16((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)), wide_tiles(rows), row_bytes(K)
    for normed in (False, True):
        graph = splash_amd.CommandGraph()
        table = add_table(graph, backend, x, weight if normed else None)
        out, beside = backend.allocate_buffer(rows * (size + 4)), backend.allocate_buffer(table_bytes(K, tiles))
        out.fill(0xA5)
        beside.fill(0xA5)
        params, source = TableParams(K, rows, tiles, 0), backend.from_array(x)
        if normed:
            graph.add("gguf_wide_table_norm_rows", [source, backend.from_array(weight), beside, out], params, (64 * -(-16 * tiles // 64), 1, 1))
        else:
            graph.add("gguf_wide_rows", [source, out], params, (rows, 1, 1))
        backend.run(graph)
        want, got = table.download(), out.download()
        assert np.array_equal(got[:rows * size].reshape(rows, size)[:, :K * 2 + K // 4], rows_of_table(want, K, rows))
        assert np.array_equal(got[rows * size:], want[tiles * (K // 256) * 9216:][:4 * rows])
        if normed:
            assert np.array_equal(beside.download(), want)


@pytest.mark.parametrize("rows,K", [(1, 256), (130, 2048), (61, 2304), (33, 8192)])
def test_rows_tables_of_norms_are_those_of_the_norm_pass(backend, rows, K):
    """GGUF_WIDE_ROWS_NORM_RMS: the experts' rows are norm_rms's to the bit, whose squares are added in another order than the
    wide table's; the wide table beside them stays what it is."""
    print(f"case rows' tables of the norm pass {rows} K={K}", flush=True)
    rng = np.random.default_rng(rows)
    x = orc.f32_to_bf16((rng.standard_normal((rows, K)) * 10.0 ** rng.integers(-2, 3, (1, K))).astype(np.float32))
    if rows > 1:
        x[0, 3], x[rows - 1, 0], x[rows // 2] = 0x7F80, 0x7FC1, 0
    weight, tiles, size = orc.f32_to_bf16((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)), wide_tiles(rows), row_bytes(K)
    source, norm = backend.from_array(x), backend.from_array(weight)
    normed, want, got = (backend.allocate_buffer(n) for n in (rows * K * 2, rows * (size + 4), rows * (size + 4)))
    beside = backend.allocate_buffer(table_bytes(K, tiles))
    for buffer in (want, got, beside):
        buffer.fill(0xA5)
    graph = splash_amd.CommandGraph()
    graph.add("norm_rms", [source, norm, normed], TableParams(K, rows, 0, 0), (rows, 1, 1))
    graph.add("gguf_wide_rows", [normed, want], TableParams(K, rows, tiles, 0), (rows, 1, 1))
    graph.add("gguf_wide_table_norm_rows", [source, norm, beside, got], TableParams(K, rows, tiles, 1), (64 * -(-16 * tiles // 64), 1, 1))
    table = add_table(graph, backend, x, weight)
    backend.run(graph)
    assert np.array_equal(got.download(), want.download())
    assert np.array_equal(beside.download(), table.download())


def gathered(backend, fmt, name, T, K, N, x, experts, selected, top_k, natives):
    """The pair's output rows of every slot, from the rows' tables and from a table of the slots."""
    rows, tiles, b = len(x), selected.size // 16 + experts, place(backend, selected, experts, top_k, T)
    images = [backend.from_array(np.concatenate([ops.pack_gguf_image(fmt, n, N, K) for n in part])) for part in natives]
    p = WideMoeParams()
    p.wide.input_size, p.wide.rows, p.wide.tiles, p.wide.out_stride, p.expert_bytes = K, rows, tiles, N, images[0].size_bytes // experts
    p.wide.cols[0], p.wide.groups = N, -(-N // 64)
    grid, source = (8 * -(-(tiles // T + experts) * p.wide.groups // 8), 1, 1), backend.from_array(x)
    by_row, by_slot, out = backend.allocate_buffer(rows * (row_bytes(K) + 4)), backend.allocate_buffer(table_bytes(K, tiles)), []
    graph = splash_amd.CommandGraph()
    graph.add("gguf_wide_rows", [source, by_row], TableParams(K, rows, tiles, 0), (rows, 1, 1))
    graph.add("gguf_wide_moe_gather", [source, b["slot_row"], b["totals"], by_slot], TableParams(K, rows, tiles, 0), (64 * -(-16 * tiles // 64), 1, 1))
    for suffix, table, more in (("x", by_row, [b["slot_row"]]), ("g", by_slot, [])):
        out.append(backend.allocate_buffer(16 * tiles * N * 2))
        out[-1].fill(0xA5)
        graph.add(f"gguf_wide_moe_{name}_t{T}_{suffix}", [images[0], images[1], table, out[-1], b["tasks"], b["totals"]] + more, p, grid)
    backend.run(graph)
    return [o.download(np.uint16).reshape(-1, N) for o in out]


@pytest.mark.parametrize("T", [2, 4, 5, 8])
@pytest.mark.parametrize("name", list(FORMATS))
def test_gathered_rows_lie_in_the_interval(backend, name, T):
    """The pair that a chunk runs, against the oracle: every slot's row is the SwiGLU of its row through its expert."""
    fmt, K, N, experts, top_k, rows = FORMATS[name], 512, 272, T + 2, 3, 700
    print(f"case wide gathered against the oracle {name} T={T}", flush=True)
    rng = np.random.default_rng(T)
    counts = [16 * height - int(rng.integers(0, 16)) for height in range(1, T + 1)] + [0]
    selected = rng.permutation(np.repeat(np.arange(experts), counts + [rows * top_k - sum(counts)]))
    _, slot_row, tasks, _ = expected_places(selected, experts, top_k, T)
    natives = [[orc.make_native(fmt, N, K, seed + e) for e in range(experts)] for seed in (1, 50)]
    x = orc.f32_to_bf16((rng.standard_normal((rows, K)) * 0.02).astype(np.float32))      # (gates of order one)
    got, _ = gathered(backend, fmt, name, T, K, N, x, experts, selected, top_k, natives)
    filled, expert_of = np.flatnonzero(slot_row != 0xFFFFFFFF), np.repeat(tasks[:, 0], 16 * tasks[:, 2].astype(np.int64))
    assert filled.size == rows * top_k
    for e in range(experts):
        at = filled[expert_of[filled] == e]
        if not len(at):
            continue
        expected = orc.swiglu(*(orc.gemm(fmt, part[e], x[slot_row[at]], N)["exact"] for part in natives))
        g, w = orc.bf16_to_f32(got[at]).astype(np.float64), orc.bf16_to_f32(expected).astype(np.float64)
        # a step of the gate's or the up value's bf16 rounding, where fp32 sums sit at its border
        assert np.all(np.abs(g - w) <= 2.0 ** -6 * np.abs(w) + 1e-6) and (got[at] != expected).mean() < 0.03


@pytest.mark.parametrize("name", list(FORMATS))
def test_gathered_rows_of_uncommon_values_give_the_slots_bits(backend, name):
    """Rows with infinities and NaN, of zeros, subnormals and the largest values, among ordinary ones that share their tiles."""
    fmt, K, N, experts, top_k, rows = FORMATS[name], 512, 144, 4, 2, 150
    print(f"case wide gathered uncommon values {name}", flush=True)
    rng = np.random.default_rng(1)
    x = orc.f32_to_bf16((rng.standard_normal((rows, K)) * 0.02).astype(np.float32))
    x[1], x[2], x[3], x[40, 5], x[41, K - 1], x[42, :3] = 0, 1, 0x7F7F, 0x7F80, 0x7FC1, (0xFF80, 0x8000, 0xFFFF)
    natives = [[orc.make_native(fmt, N, K, seed + e) for e in range(experts)] for seed in (1, 50)]
    by_row, by_slot = gathered(backend, fmt, name, 4, K, N, x, experts, rng.integers(0, experts, rows * top_k), top_k, natives)
    assert np.array_equal(by_row, by_slot)
    values = orc.bf16_to_f32(by_row)
    assert np.isnan(values).any() and (np.abs(values) < 10).any()
