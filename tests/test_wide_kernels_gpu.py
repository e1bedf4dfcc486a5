"""GPU tests of a prompt chunk's kernels one by one, dispatched with the parameters their operators would give them
(ops::Linear::addWide*, ops::MoE::addChunk, ops::PagedAttention::addPrompt*): the wide table, every tile height of the wide
projection, the grouping of a chunk's routes over several windows, the experts' tiles, and the attention of a chunk's blocks,
against the oracle and 64-bit sums."""
import ctypes

import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc
from tests.test_attention_gpu import build_context, tolerance
from tests.test_gguf_gpu import check_interval, run_projection

pytestmark = pytest.mark.gpu

FORMATS = {"q4k": ops.FMT_Q4K, "q5k": ops.FMT_Q5K, "q6k": ops.FMT_Q6K}
U = ctypes.c_uint32


class TableParams(ctypes.Structure):
    _fields_ = [(n, U) for n in ("input_size", "rows", "tiles", "reserved")]


class WideParams(ctypes.Structure):
    _fields_ = [(n, U) for n in ("input_size", "rows", "tiles", "row_groups", "splits", "out_stride", "groups")] + \
               [("cols", U * 3), ("offset", U * 3), ("reserved", U * 3)]


class ReduceParams(ctypes.Structure):
    _fields_ = [(n, U) for n in ("rows", "columns", "splits", "reserved")]


class WideMoeParams(ctypes.Structure):
    _fields_ = [("wide", WideParams), ("expert_bytes", ctypes.c_uint64), ("reserved", ctypes.c_uint64)]


class ChunkParams(ctypes.Structure):
    _fields_ = [(n, U) for n in ("routes", "experts", "top_k", "task_tiles")]


class Sequence(ctypes.Structure):
    _fields_ = [("first_row", U), ("committed", U), ("table_first", U), ("rows", ctypes.c_uint16), ("steps_per_split", ctypes.c_uint16)]


class AttentionParams(ctypes.Structure):
    _fields_ = [(n, U) for n in ("q_heads", "kv_heads", "head_dim", "rotary_pairs", "normalize", "qkv_stride", "splits", "sequences",
                                 "table_tiles", "gated", "int8_queries", "chunk_rows")] + [("page_bytes", ctypes.c_uint64), ("sequence", Sequence * 8)]


assert [ctypes.sizeof(t) for t in (TableParams, WideParams, ReduceParams, WideMoeParams, ChunkParams, AttentionParams)] == [16, 64, 16, 80, 16, 184]


def wide_tiles(rows):
    return (rows + 127) // 128 * 8


def tile_bytes(K):
    return K // 256 * 9 * 1024


def table_bytes(K, tiles):
    return tiles * tile_bytes(K) + tiles * 64


def add_table(graph, backend, x_bits, weight=None):
    """The wide table of bf16 rows (of their norm, with a weight)."""
    rows, K = x_bits.shape
    tiles = wide_tiles(rows)
    table = backend.allocate_buffer(table_bytes(K, tiles))
    table.fill(0xA5)
    name = "gguf_wide_table_norm" if weight is not None else "gguf_wide_table" if K <= 8192 else "gguf_wide_table_long"
    x = backend.from_array(x_bits)
    graph.add(name, [x, backend.from_array(weight) if weight is not None else x, table], TableParams(K, rows, tiles, 0),
              (64 * ((16 * tiles + 63) // 64), 1, 1))
    return table


def rows_of(rng, rows, K):
    """bf16 rows of different sizes, one of zeros, one with an entry far above the others."""
    x = rng.standard_normal((rows, K)).astype(np.float32) * np.float32(2.0) ** rng.integers(-12, 12, (rows, 1)).astype(np.float32)
    x[rows // 2] = 0
    x[-1, K // 3] = 300 * np.abs(x[-1]).max()
    return orc.f32_to_bf16(x)


@pytest.mark.parametrize("K,norm", [(256, False), (2304, False), (2304, True), (8192, False), (8192, True), (8448, False), (32768, False)])
def test_the_wide_table_holds_its_rows(backend, K, norm):
    """Every operand times its row's scale is the row's bf16 value, and the three parts of a group's sum add up to it, for
    widths that fill a thread's registers and widths that end inside them; rows past the last are zeros."""
    print(f"case wide table K={K} norm={norm}", flush=True)
    rng = np.random.default_rng(K)
    rows = 21
    x = rows_of(rng, rows, K)
    weight = orc.f32_to_bf16((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)) if norm else None
    graph = splash_amd.CommandGraph()
    table = add_table(graph, backend, x, weight)
    backend.run(graph)
    tiles = wide_tiles(rows)
    raw = table.download(np.uint8)
    values = raw[:tiles * tile_bytes(K)].view(np.uint16).reshape(tiles, K // 256, 9, 64, 8)
    scale = raw[tiles * tile_bytes(K):].view(np.float32).astype(np.float64)
    got = orc.table_rows(np.ascontiguousarray(values[:, :, :8]), K, tiles).view(np.float16).astype(np.float64)
    assert not got[rows:].any()
    largest = np.abs(got[:rows]).max(axis=1)
    assert np.all((largest == 0) | ((largest >= 2.0 ** 14) & (largest < 2.0 ** 15)))
    assert np.array_equal(np.exp2(np.rint(np.log2(scale[:rows]))), scale[:rows])
    back = orc.f32_to_bf16((got * scale[:, None])[:rows].astype(np.float32))
    want = x if weight is None else orc.rms_norm(x, weight)
    if weight is None:
        assert np.array_equal(back & 0x7FFF, want & 0x7FFF) and np.array_equal(back[want != 0x8000], want[want != 0x8000])
    else:      # the sum of squares is taken in another order: a step of bf16 now and then
        apart = np.abs(back.astype(np.int64) - want.astype(np.int64))
        assert apart.max() <= 1 and (apart > 0).mean() < 5e-3, (apart.max(), (apart > 0).mean())
    parts = values[:, :, 8].view(np.float16).astype(np.float64).reshape(tiles, K // 256, 4, 16, 8)      # [t][block][part][r][group]
    sums = parts.sum(axis=2).transpose(0, 2, 1, 3).reshape(tiles * 16, K // 32) * 32
    groups = got.reshape(tiles * 16, K // 32, 32)
    assert not parts[:, :, 3].any()
    # an fp32 sum of 32 terms, and what three fp16 parts of it leave (33 bits, or fp16's smallest step)
    assert np.all(np.abs(sums - groups.sum(axis=2)) <= 32 * 2.0 ** -24 * np.abs(groups).sum(axis=2) + 2.0 ** -19)


def project(backend, name, images, cols, table, out, rows, K, T, splits=1, residual=None, columns=128, stride=None):
    """One dispatch of gguf_wide_<name>: the row tiles dealt over as few workgroups as hold them."""
    offset = np.concatenate([[0], np.cumsum(cols)])[:len(cols)]
    p = WideParams(K, rows, wide_tiles(rows), -(-((rows + 15) // 16) // T), splits, stride or int(sum(cols)), sum(-(-n // columns) for n in cols))
    for s, n in enumerate(cols):
        p.cols[s], p.offset[s] = n, int(offset[s])
    images = (images + images[-1:] * 2)[:3]
    graph = splash_amd.CommandGraph()
    items = p.row_groups * splits * p.groups
    graph.add(f"gguf_wide_{name}", images + [table, out, residual or table], p, (8 * -(-items // 8), 1, 1))
    backend.run(graph)


@pytest.mark.parametrize("T", [4, 6, 7, 8])
@pytest.mark.parametrize("name", list(FORMATS))
def test_every_tile_height_lies_in_the_interval(backend, name, T):
    """Row tiles that fill a workgroup's height, leave it short and are dealt unevenly over two, tensors that end inside a
    column group, K whole and in parts, the plain, residual, split and gate/up epilogues: fp32 results within the reference's
    bound of the 64-bit dot and on the whole no further from it than the decode kernels', the bf16 ones their roundings."""
    fmt, K, cols = FORMATS[name], 768, [144, 128, 16]
    print(f"case wide projection {name} T={T}", flush=True)
    rng = np.random.default_rng(T)
    N, linear = sum(cols), ops.Linear(backend)
    natives = [orc.make_native(fmt, n, K, 10 * T + n) for n in cols]
    images = [backend.from_array(ops.pack_gguf_image(fmt, native, n, K)) for native, n in zip(natives, cols)]
    for rows in (3, 16 * T - 15, 16 * (2 * T - 1) - 5):
        x = rows_of(rng, rows, K)
        residual = orc.f32_to_bf16(rng.standard_normal((rows, N)).astype(np.float32))
        want = [orc.gemm(fmt, native, x, n) for native, n in zip(natives, cols)]
        want = {key: np.concatenate([w[key] for w in want], axis=1) for key in ("exact", "bound")}
        graph = splash_amd.CommandGraph()
        table, res = add_table(graph, backend, x), backend.from_array(residual)
        backend.run(graph)
        decode, _, _ = run_projection(backend, linear, fmt, list(zip(cols, natives)), K, x, float32=True)
        far = lambda got: np.sqrt((((got - want["exact"]) / np.maximum(want["bound"], 1e-300)) ** 2).mean())
        for splits in (1, 3):
            partials = backend.allocate_buffer(splits * rows * N * 4)
            partials.fill(0xFF)
            project(backend, f"{name}_t{T}_p", images, cols, table, partials, rows, K, T, splits)
            outs = {}
            for kind, size in (("f32", 4), ("a", 2), ("r", 2)):
                outs[kind] = backend.allocate_buffer(rows * N * size)
                graph = splash_amd.CommandGraph()
                graph.add(f"gguf_wide_reduce_{kind}", [partials, outs[kind], res], ReduceParams(rows, N, splits, 0), (-(-rows * N // 1024), 1, 1))
                backend.run(graph)
            f32 = outs["f32"].download(np.float32).reshape(rows, N)
            assert np.all(np.abs(f32.astype(np.float64) - want["exact"]) <= want["bound"])
            print(f"  rows {rows} parts {splits}: rms error over the bound {far(f32):.3e}, decode kernels {far(decode):.3e}", flush=True)
            assert far(f32) <= far(decode)
            rounded = orc.f32_to_bf16(f32), orc.f32_to_bf16(f32 + orc.bf16_to_f32(residual))
            for kind, expected in zip(("a", "r"), rounded):
                assert np.array_equal(outs[kind].download(np.uint16).reshape(rows, N), expected)
            if splits == 1:
                for kind, expected in zip(("a", "r"), rounded):
                    outs[kind].fill(0xFF)
                    project(backend, f"{name}_t{T}_{kind}", images, cols, table, outs[kind], rows, K, T, residual=res)
                    assert np.array_equal(outs[kind].download(np.uint16).reshape(rows, N), expected)
                # a gate/up pair: the first tensor's columns against themselves shifted
                n = 112
                up = backend.from_array(ops.pack_gguf_image(fmt, natives[0][32 * len(natives[0]) // 144:], n, K))
                pair = backend.allocate_buffer(rows * n * 2)
                project(backend, f"{name}_t{T}_g", [images[0], up], [n], table, pair, rows, K, T, columns=64)
                expected = orc.swiglu(f32[:, :n], f32[:, 32:32 + n])
                got = pair.download(np.uint16).reshape(rows, n)
                g, w = orc.bf16_to_f32(got).astype(np.float64), orc.bf16_to_f32(expected).astype(np.float64)
                assert np.all(np.abs(g - w) <= 2.0 ** -7 * np.abs(w) + 1e-38) and (got != expected).mean() < 0.03      # (exp2's last bit)


@pytest.mark.parametrize("T", [6, 7, 8])
@pytest.mark.parametrize("name", ["q4k", "q6k", "staged_q4k"])
def test_tail_columns_in_shorter_workgroups_change_nothing(backend, name, T):
    """The last column groups in workgroups of four row tiles, one group to all but one of them, tensors that end inside a
    group, rows that leave the last workgroup short: every epilogue's bits are those of the same columns in tall ones."""
    fmt, K, cols = FORMATS[name[-3:]], 768, [144, 128, 16]
    if name.startswith("staged"):
        if T < 8:
            pytest.skip("the staged rule has the tallest tile alone")
        cols = [256, 128, 128]
    print(f"case wide tail {name} T={T}", flush=True)
    rng = np.random.default_rng(T)
    N = sum(cols)
    images = [backend.from_array(ops.pack_gguf_image(fmt, orc.make_native(fmt, n, K, 10 * T + n), n, K)) for n in cols]
    for rows in (5, 16 * (2 * T - 1) - 5):
        residual = backend.from_array(orc.f32_to_bf16(rng.standard_normal((rows, N)).astype(np.float32)))
        graph = splash_amd.CommandGraph()
        table = add_table(graph, backend, rows_of(rng, rows, K))
        backend.run(graph)
        tiles = (rows + 15) // 16
        for kind, size, widths, columns in (("p", 4, cols, 128), ("a", 2, cols, 128), ("r", 2, cols, 128), ("g", 2, cols[1:2], 64)):
            weights = images if kind != "g" else [images[1], images[1]]
            groups, span, got = sum(-(-n // columns) for n in widths), sum(widths), []
            for tail in (0, 1, groups - 1):
                p = WideParams(K, rows, wide_tiles(rows), -(-tiles // T), 1, span, groups)
                for s, n in enumerate(widths):
                    p.cols[s], p.offset[s] = n, sum(widths[:s])
                p.reserved[0], p.reserved[1] = tail, -(-tiles // 4)
                out = backend.allocate_buffer(rows * span * size)
                out.fill(0xFF)
                graph = splash_amd.CommandGraph()
                blocks = 8 * -(-p.row_groups * (groups - tail) // 8) + 8 * -(-p.reserved[1] * tail // 8)
                graph.add(f"gguf_wide_{name}_t{T}_{kind}", (weights + weights[-1:] * 2)[:3] + [table, out, residual], p, (blocks, 1, 1))
                backend.run(graph)
                got.append(out.download(np.uint8).tobytes())
            assert got[1] == got[0] and got[2] == got[0], (kind, rows)


@pytest.mark.parametrize("name", list(FORMATS))
def test_a_staged_projection_lies_in_the_staged_interval(backend, name):
    """The staged rule's tile, K whole and in parts."""
    fmt, K, N, rows = FORMATS[name], 768, 272, 203
    print(f"case wide staged {name}", flush=True)
    x = rows_of(np.random.default_rng(5), rows, K)
    native = orc.make_native(fmt, N, K, 3)
    image, want = backend.from_array(ops.pack_gguf_image(fmt, native, N, K)), orc.gemm_staged(fmt, native, x, N)
    graph = splash_amd.CommandGraph()
    table = add_table(graph, backend, x)
    backend.run(graph)
    for splits in (1, 3):
        partials = backend.allocate_buffer(splits * rows * N * 4)
        project(backend, f"staged_{name}_t8_p", [image], [N], table, partials, rows, K, 8, splits)
        got = partials.download(np.float32).reshape(splits, rows, N).astype(np.float64).sum(axis=0)
        distance = np.abs(got - want["staged"].astype(np.float64))
        assert np.all(distance <= want["accumulation"] + np.abs(want["staged"]) * 2.0 ** -23), float((distance / want["accumulation"]).max())


def place(backend, selected, experts, top_k, T):
    """moe_chunk_count and moe_chunk_place over the routes; their buffers."""
    routes = selected.size
    windows, tiles = -(-routes // 2048), routes // 16 + min(experts, routes)
    b = dict(selected=backend.from_array(selected.astype(np.uint32)), counts=backend.allocate_buffer(windows * experts * 4),
             route_slot=backend.allocate_buffer(routes * 4), slot_row=backend.allocate_buffer(tiles * 64),
             tasks=backend.allocate_buffer((tiles // 2 + experts) * 16), totals=backend.allocate_buffer(16))
    for buffer in list(b.values())[1:]:
        buffer.fill(0xEE)
    p, graph = ChunkParams(routes, experts, top_k, T), splash_amd.CommandGraph()
    graph.add("moe_chunk_count", [b["selected"], b["counts"]], p, (windows, 1, 1), (1024, 1, 1))
    graph.add("moe_chunk_place", [b[n] for n in ("selected", "counts", "route_slot", "slot_row", "tasks", "totals")], p, (windows, 1, 1), (1024, 1, 1))
    backend.run(graph)
    return b


def expected_places(selected, experts, top_k, T):
    """Slots, slot rows and tasks as abi/Moe.h states them."""
    route_slot, slot_row, tasks, tile = np.zeros(selected.size, np.int64), [], [], 0
    for e in range(experts):
        mine = np.flatnonzero(selected == e)
        count = -(-len(mine) // 16)
        route_slot[mine] = 16 * tile + np.arange(len(mine))
        slot_row += list(mine // top_k) + [0xFFFFFFFF] * (16 * count - len(mine))
        parts = -(-count // T)
        tasks += [(e, tile + count * i // parts, count * (i + 1) // parts - count * i // parts) for i in range(parts)]
        tile += count
    return route_slot, np.array(slot_row, np.uint32), np.array(tasks, np.uint32), tile


def skewed(rng, routes, experts):
    """Routes of which the first expert takes many, some none, the last a few."""
    weights = rng.random(experts) ** 4
    weights[0], weights[experts // 2] = weights.sum(), 0
    selected = rng.choice(experts, routes, p=weights / weights.sum())
    selected[[0, routes - 1]] = experts - 1
    return selected


@pytest.mark.parametrize("rows,top_k,experts,T", [(1, 1, 2, 2), (256, 8, 128, 4), (257, 8, 128, 5), (640, 9, 80, 5), (2048, 9, 129, 5), (2048, 16, 256, 4),
                                                  (2048, 8, 128, 8)])
def test_a_chunks_routes_are_placed_across_windows(backend, rows, top_k, experts, T):
    """One window of 2048 routes, one route more, several, the last one short: every route's slot follows those of the windows
    before it, an expert's slots are whole tiles, its tasks even."""
    print(f"case moe place rows={rows} top_k={top_k} experts={experts}", flush=True)
    selected = skewed(np.random.default_rng(rows + experts), rows * top_k, experts)
    b = place(backend, selected, experts, top_k, T)
    route_slot, slot_row, tasks, tiles = expected_places(selected, experts, top_k, T)
    assert list(b["totals"].download(np.uint32)[:2]) == [tiles, len(tasks)]
    assert np.array_equal(b["route_slot"].download(np.uint32), route_slot)
    assert np.array_equal(b["slot_row"].download(np.uint32)[:16 * tiles], slot_row)
    assert np.array_equal(b["tasks"].download(np.uint32).reshape(-1, 4)[:len(tasks), :3], tasks)


@pytest.mark.parametrize("T", [2, 4, 5])
@pytest.mark.parametrize("name", list(FORMATS))
def test_expert_tiles_lie_in_the_interval(backend, name, T):
    """The experts' projections over gathered rows and over the slots' own, tasks of every height up to T, two windows of
    routes, columns that end inside a column group: each slot's row in the interval of its row through its expert."""
    fmt, K, N, experts, top_k, rows = FORMATS[name], 512, 272, T + 2, 3, 700
    print(f"case wide experts {name} T={T}", flush=True)
    rng = np.random.default_rng(T)
    routes = rows * top_k
    # an expert of each height, its last tile short; one without a row; one of many tasks with the routes left
    counts = [16 * height - int(rng.integers(0, 16)) for height in range(1, T + 1)] + [0]
    selected = rng.permutation(np.repeat(np.arange(experts), counts + [routes - sum(counts)]))
    b = place(backend, selected, experts, top_k, T)
    route_slot, slot_row, tasks, live = expected_places(selected, experts, top_k, T)
    assert set(tasks[:, 2]) == set(range(1, T + 1)) and len(tasks) >= T + 3
    tiles = routes // 16 + experts
    gate, up = ([orc.make_native(fmt, N, K, seed + e) for e in range(experts)] for seed in (1, 50))
    image_of = lambda natives: backend.from_array(np.concatenate([ops.pack_gguf_image(fmt, n, N, K) for n in natives]))
    images = image_of(gate), image_of(up)
    x = orc.f32_to_bf16((rng.standard_normal((rows, K)) * 0.02).astype(np.float32))      # (gates of order one)
    slots = np.zeros((16 * tiles, K), np.uint16)
    filled = np.flatnonzero(slot_row != 0xFFFFFFFF)
    slots[filled] = x[slot_row[filled]]
    expert_of = np.repeat(tasks[:, 0], 16 * tasks[:, 2].astype(np.int64))      # of each live slot
    p = WideMoeParams()
    p.wide.input_size, p.wide.tiles, p.wide.out_stride, p.expert_bytes = K, tiles, N, images[0].size_bytes // experts
    p.wide.cols[0] = N
    want = {}
    for e in range(experts):
        at = filled[expert_of[filled] == e]
        if len(at):
            want[e] = at, orc.gemm(fmt, gate[e], slots[at], N), orc.gemm(fmt, up[e], slots[at], N)
    assert sum(len(at) for at, _, _ in want.values()) == routes
    for table_kernel, source in (("gguf_wide_moe_gather", x), ("gguf_wide_moe_rows", slots)):
        table, out = backend.allocate_buffer(table_bytes(K, tiles)), backend.allocate_buffer(16 * tiles * N * 2)
        table.fill(0xA5)
        for suffix, span in (("a", 128), ("g", 64)):
            p.wide.groups = -(-N // span)
            graph = splash_amd.CommandGraph()
            graph.add(table_kernel, [backend.from_array(source), b["slot_row"], b["totals"], table], TableParams(K, len(source), tiles, 0),
                      (64 * -(-16 * tiles // 64), 1, 1))
            graph.add(f"gguf_wide_moe_{name}_t{T}_{suffix}", [images[0], images[1], table, out, b["tasks"], b["totals"]], p,
                      (8 * -(-(tiles // T + experts) * p.wide.groups // 8), 1, 1))
            backend.run(graph)
            got = out.download(np.uint16).reshape(-1, N)
            for at, first, second in want.values():
                if suffix == "a":
                    check_interval(orc.bf16_to_f32(got[at]), first)
                else:
                    expected = orc.swiglu(first["exact"], second["exact"])
                    g, w = orc.bf16_to_f32(got[at]).astype(np.float64), orc.bf16_to_f32(expected).astype(np.float64)
                    # a step of the gate's or the up value's bf16 rounding, where fp32 sums sit at its border
                    assert np.all(np.abs(g - w) <= 2.0 ** -6 * np.abs(w) + 1e-6) and (got[at] != expected).mean() < 0.03


@pytest.mark.parametrize("name", list(FORMATS))
def test_expert_tiles_of_tall_tasks_lie_in_the_interval(backend, name):
    """The same of tasks of up to eight row tiles, whose kernels hold a body for each height of four and more."""
    test_expert_tiles_lie_in_the_interval(backend, name, 8)


def test_the_conversion_to_bf16_is_the_integer_rule(backend):
    """Round to nearest even of every upper half with lower halves at a tie and beside it, at the ends and between: zeros,
    subnormals, every exponent's carries, the overflow to infinity, infinities and NaN payloads."""
    print("case bf16 conversion", flush=True)
    lower = np.array([0, 1, 0x4000, 0x7FFF, 0x8000, 0x8001, 0xC000, 0xFFFF], np.uint32)
    values = ((np.arange(1 << 16, dtype=np.uint32) << 16)[:, None] | lower).view(np.float32)
    out = backend.allocate_buffer(values.size * 2)
    graph = splash_amd.CommandGraph()
    graph.add("gguf_wide_reduce_a", [backend.from_array(values), out, out], ReduceParams(*values.shape, 1, 0), (values.size // 1024, 1, 1))
    backend.run(graph)
    assert np.array_equal(out.download(np.uint16), orc.f32_to_bf16(values).ravel())


# half a wave's piece, one and a half, three and a half, and the four that a wave holds
@pytest.mark.parametrize("K", [256, 768, 1792, 2048])
@pytest.mark.parametrize("kind", ["gather", "rows"])
def test_slots_tables_by_the_tile_are_those_by_the_row(backend, K, kind):
    """The slots' tables put together in LDS and those that the rows write are the same bytes: rows of ordinary values, of
    zeros, subnormals and the largest ones, with infinities and NaN, empty slots, and tiles past the count left alone."""
    print(f"case slot tables by the tile {kind} K={K}", flush=True)
    rng = np.random.default_rng(K)
    tiles, live, rows = 7, 5, 61
    slots = 16 * tiles
    source = orc.f32_to_bf16((rng.standard_normal((rows if kind == "gather" else slots, K)) * 10.0 ** rng.integers(-6, 7, (1, K))).astype(np.float32))
    source[1], source[2], source[3] = 0, 1, 0x7F7F
    source[4, 5], source[5, K - 1], source[6, :3] = 0x7F80, 0x7FC1, (0xFF80, 0x8000, 0xFFFF)
    slot_row = np.where(rng.random(slots) < 0.2, 0xFFFFFFFF, rng.integers(0, rows, slots)).astype(np.uint32)
    slot_row[:7] = np.arange(7)
    x, s, totals = backend.from_array(source), backend.from_array(slot_row), backend.from_array(np.array([live, 0, 0, 0], np.uint32))
    got = []
    for suffix, grid, threads in (("", 64 * -(-slots // 64), 256), ("_tile", tiles, 1024)):
        table = backend.allocate_buffer(table_bytes(K, tiles))
        table.fill(0xA5)
        graph = splash_amd.CommandGraph()
        graph.add(f"gguf_wide_moe_{kind}{suffix}", [x, s, totals, table], TableParams(K, len(source), tiles, 0), (grid, 1, 1), (threads, 1, 1))
        backend.run(graph)
        got.append(table.download())
    assert np.array_equal(got[0], got[1]) and (got[0] != 0xA5).any()


# head counts that end inside a workgroup's group of heads, every kind of rotation, a ragged last block
@pytest.mark.parametrize("geometry,pairs,gated,normalize", [((64, 8, 128), 64, False, True), ((6, 2, 128), 32, True, True), ((3, 1, 128), 0, False, True),
                                                            ((8, 8, 128), 8, True, False), ((16, 8, 64), 32, False, True), ((9, 3, 64), 24, True, True)])
def test_a_chunks_heads_by_vectors_are_those_by_rows(backend, geometry, pairs, gated, normalize):
    """attention_q8_qkv_vectors leaves the bytes of attention_q8_qkv_rows: queries, their sums, keys, values and scales, with
    rows of zeros, of large values and of an infinity and a NaN."""
    q_heads, kv_heads, D = geometry
    print(f"case heads by vectors {geometry} pairs={pairs} gated={gated} normalize={normalize}", flush=True)
    rng = np.random.default_rng(q_heads + pairs)
    tokens, committed, first = 45, 250, 3
    blocks = -(-tokens // 16)
    width = ((2 if gated else 1) * q_heads + 2 * kv_heads) * D
    qkv = orc.f32_to_bf16(rng.standard_normal((first + tokens, width)).astype(np.float32) * 2)
    qkv[first + 1] = 0
    qkv[first + 2] = orc.f32_to_bf16(np.full(width, 2.0 ** 60, np.float32))
    qkv[first + 3, 5], qkv[first + 4, D - 1] = 0x7F80, 0x7FC0    # (of the first query head: a key head's scale is a comparison)
    weights = [orc.f32_to_bf16((1 + 0.1 * rng.standard_normal(D)).astype(np.float32)) for _ in range(2)]
    angles = rng.uniform(0, 6.28, (first + tokens, max(pairs, 1))).astype(np.float32)
    inputs = [backend.from_array(a) for a in (qkv, *weights, np.cos(angles), np.sin(angles))]
    pages = -(-(committed + tokens) // ops.PAGE_TOKENS)
    table = backend.from_array(rng.permutation(pages).astype(np.uint64))
    p = AttentionParams(q_heads, kv_heads, D, pairs, normalize, width, 1, blocks, 0, gated, 0, tokens, ops.kv_page_bytes(kv_heads, D))
    s = p.sequence[0]
    s.first_row, s.committed, s.table_first, s.rows, s.steps_per_split = first, committed, 0, 16, 1
    got = []
    for name, grid in (("rows", q_heads + kv_heads), ("vectors", -(-q_heads // (512 // D)) + kv_heads)):
        out = [backend.from_array(np.full(n, 0xA5, np.uint8)) for n in (blocks * q_heads * 16 * D * 2, blocks * q_heads * 16 * 4, pages * p.page_bytes)]
        graph = splash_amd.CommandGraph()
        graph.add(f"attention_q8_qkv_{name}_d{D}", [*inputs, *out[:2], table, out[2]], p, (grid, blocks, 1))
        backend.run(graph)
        queries, sums, pool = out[0].download(np.uint16).copy(), out[1].download(np.uint32).copy(), out[2].download()
        for values, low, mask in ((queries, 0x7C00, 0x7FFF), (sums, 0x7F800000, 0x7FFFFFFF)):    # (one NaN is as good as another)
            values[(values & mask) > low] = low + 1
        got.append((queries, sums, pool))
    assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("geometry,tokens,committed,gated", [((64, 8, 128), 200, 300, False), ((64, 8, 128), 53, 0, True), ((32, 8, 128), 200, 250, True),
                                                             ((32, 8, 128), 64, 1000, False), ((16, 8, 64), 200, 300, False), ((16, 8, 64), 37, 700, True)])
def test_a_chunks_blocks_attend_whole_histories(backend, geometry, tokens, committed, gated):
    """The prompt attention: both prepare kernels store the oracle's keys and values; a block's whole history in a workgroup,
    and in splits, lies as close to the 64-bit softmax as the chunked plan's rows, with and without output gates, for every
    compiled group of heads."""
    q_heads, kv_heads, D = geometry
    print(f"case prompt attention {geometry} tokens={tokens} committed={committed} gated={gated}", flush=True)
    rng = np.random.default_rng(tokens + committed + D)
    pairs, blocks, group = D // 4, -(-tokens // 16), q_heads // kv_heads
    kv, logical, table = build_context(rng, backend, q_heads, kv_heads, D, tokens, committed)
    start = kv.download()
    width = ((2 if gated else 1) * q_heads + 2 * kv_heads) * D
    qkv = orc.f32_to_bf16(rng.standard_normal((tokens, width)).astype(np.float32))
    qw, kw = (orc.f32_to_bf16((1 + 0.1 * rng.standard_normal(D)).astype(np.float32)) for _ in range(2))
    angles = rng.uniform(0, 6.28, (tokens, pairs)).astype(np.float32)
    cosv, sinv = np.cos(angles).astype(np.float32), np.sin(angles).astype(np.float32)
    tree = ops.chain_tree_rows([min(16, tokens - first) for first in range(0, tokens, 16)])
    bufs = [backend.from_array(a) for a in (qkv, qw, kw, cosv, sinv)]
    tree_buf = backend.from_array(tree)
    # the oracle: every row stored, then every block
    heads = qkv[:, :2 * q_heads * D].reshape(tokens, q_heads, 2, D) if gated else None
    plain = np.concatenate([heads[:, :, 0].reshape(tokens, -1), qkv[:, 2 * q_heads * D:]], axis=1) if gated else qkv
    kc, ks, vc, vs = (a.copy() for a in logical)
    q, kf, vf = orc.attention_prepare(q_heads, kv_heads, D, plain, qw, kw, cosv, sinv, pairs)
    kcod, kscl = orc.kv_quantize(kf)
    vcod, vscl = orc.kv_quantize(vf)
    for r in range(tokens):
        page, s = table[(committed + r) // ops.PAGE_TOKENS], (committed + r) % ops.PAGE_TOKENS
        kc[page, :, s], ks[page, :, s], vc[page, :, s], vs[page, :, s] = kcod[r], kscl[r], vcod[r], vscl[r]
    want = []
    for first in range(0, tokens, 16):
        rows = min(16, tokens - first)
        anc = tree["ancestors"][first:first + rows].astype(np.uint32)
        want.append(orc.attention(np.ascontiguousarray(q[first:first + rows]), kc, ks, vc, vs, table, anc, committed + first)[1])
    want = np.concatenate(want)
    if gated:
        want = want / (1 + np.exp(-orc.bf16_to_f32(heads[:, :, 1]).astype(np.float64)))
    error, rows_of_label = {}, {}

    def check(label, out):
        got = out.download(np.uint16).reshape(tokens, q_heads, D)
        cos, err = tolerance(got, want)
        assert cos >= 0.9999 and err < 0.02, (label, cos, err)
        error[label] = float(np.sqrt(((orc.bf16_to_f32(got) - want) ** 2).mean()))
        rows_of_label[label] = got
        for a, b in zip(kv.unpack_pages(kv.download()), (kc, ks, vc, vs)):
            assert np.array_equal(a[table], b[table]), label
    plan = ops.AttentionChunkPlan(q_heads, kv_heads, D, [(0, tokens, committed, 0)], rotary_pairs=pairs, normalize=True, gated=gated)
    sizes = plan.workspace_sizes()
    ws = type("Workspace", (), dict(zip(("queries", "query_sums", "partials", "partial_sums"), map(backend.allocate_buffer, sizes))))
    out = backend.allocate_buffer(tokens * q_heads * D * 2)
    graph = splash_amd.CommandGraph()
    ops.PagedAttention.add_chunk_projection(graph, plan, bufs[0], ws, kv, query_norm=bufs[1], key_norm=bufs[2], rope_cos=bufs[3], rope_sin=bufs[4])
    ops.PagedAttention.add_chunk_attention(graph, plan, ws, tree_buf, kv, out, packed_qkv=bufs[0] if gated else None)
    backend.run(graph)
    check("chunked", out)
    steps = -(-(committed + tokens) // 64)
    name = f"_d{D}_g{group}"
    for prepare, splits in (("rows", 1), ("chunk", 1), ("rows", 3)):
        kv.upload(start)
        queries, sums = backend.allocate_buffer(blocks * q_heads * 16 * D * 2), backend.allocate_buffer(blocks * q_heads * 64)
        queries.fill(0xFF)
        per = -(-steps // splits)
        p = AttentionParams(q_heads, kv_heads, D, pairs, 1, width, -(-steps // per), blocks, 0, int(gated), 0, tokens, kv.page_bytes)
        p.sequence[0] = Sequence(0, committed, 0, 16, per)
        graph, out = splash_amd.CommandGraph(), backend.allocate_buffer(tokens * q_heads * D * 2)
        graph.add(f"attention_q8_qkv_{prepare}_d{D}", bufs + [queries, sums, kv.table, kv.pool], p,
                  (q_heads + kv_heads, blocks, 1) if prepare == "rows" else (q_heads + kv_heads, 16, blocks), (256 if prepare == "rows" else D, 1, 1))
        inputs = [queries, sums, tree_buf, kv.table, kv.pool]
        if p.splits == 1:
            graph.add("attention_q8_whole" + name, inputs + [out, bufs[0] if gated else out], p, (kv_heads * blocks, 1, 1))
        else:
            partials = backend.allocate_buffer(blocks * q_heads * 16 * p.splits * D * 2)
            partial_sums = backend.allocate_buffer(blocks * q_heads * 16 * p.splits * 8)
            graph.add("attention_q8_split_chunk" + name, inputs + [partials, partial_sums], p, (kv_heads, p.splits, blocks))
            graph.add(f"attention_reduce_chunk_d{D}", [partials, partial_sums, out, out, bufs[0] if gated else out], p, (q_heads, 16, blocks))
        backend.run(graph)
        check(f"{prepare} {p.splits}", out)
    print("  rms error: " + ", ".join(f"{k} {v:.3e}" for k, v in error.items()), flush=True)
    assert all(v <= 1.01 * error["chunked"] for v in error.values())
    assert np.array_equal(rows_of_label["rows 1"], rows_of_label["chunk 1"])      # the two prepare kernels stage the same bytes
