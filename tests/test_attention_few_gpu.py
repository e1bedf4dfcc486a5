"""attention_q8_few against attention_q8_split: the same partials bit for bit, whatever the rows, the parts and the history."""
import numpy as np
import pytest

import splash_amd
from splash_amd import ops, synthetic
from tests import oracle as orc
from tests.test_wide_kernels_gpu import AttentionParams, Sequence

pytestmark = pytest.mark.gpu


def _tree(rng, counts):
    """Tree rows of random trees: a row's ancestors are itself and a random earlier row's."""
    out = []
    for rows in counts:
        masks = [1]
        for r in range(1, rows):
            masks.append(masks[int(rng.integers(0, r))] | 1 << r)
        out += [(m, 0) for m in masks]
    return np.array(out, np.uint32)


def _partials(backend, kernel, parts, threads, heads, lanes, tree, pages, steps_per_split):
    Q, K, D = heads
    splits = max(-(-(-(-(c + r) // 64)) // steps_per_split) for c, r in lanes)
    p = AttentionParams(Q, K, D, 0, 0, (Q + 2 * K) * D, splits, len(lanes), 0, 0, 0, 0, pages["kv"].page_bytes)
    first = 0
    for i, (committed, rows) in enumerate(lanes):
        p.sequence[i] = Sequence(first, committed, pages["first"][i], rows, steps_per_split)
        first += rows
    n = len(lanes) * Q * 16 * splits
    out, sums = backend.from_array(np.full(n * D, 0x7E00, np.uint16)), backend.from_array(np.full(2 * n, 0x7FC00000, np.uint32))
    graph = splash_amd.CommandGraph()
    graph.add(kernel, [pages["queries"], pages["sums"], tree, pages["kv"].table, pages["kv"].pool, out, sums], p, (K * parts, splits, len(lanes)), (threads, 1, 1))
    backend.run(graph)
    shape = (len(lanes), K, splits, Q // K, 16)
    o, s = out.download(np.uint16).reshape(*shape, D), sums.download(np.uint32).reshape(*shape, 2)
    return [(o[i, :, :, :, :rows], s[i, :, :, :, :rows]) for i, (_, rows) in enumerate(lanes)]


LANES = {
    "empty": [(0, 1)],
    "two rows": [(63, 2)],
    "page edges": [(255, 2), (256, 1), (257, 2)],
    "three rows": [(1000, 3), (61, 1)],
    "eight": [(2049, 8), (640, 5), (0, 7)],
    "long": [(9999, 1)],
}


@pytest.mark.parametrize("heads", [(64, 8, 128), (32, 8, 128), (16, 8, 64)], ids=["g8", "g4", "d64"])
@pytest.mark.parametrize("case", list(LANES))
def test_few_rows_equal_the_split_kernel(backend, heads, case):
    Q, K, D = heads
    G, lanes = Q // K, LANES[case]
    rng = np.random.default_rng(7)
    counts = [-(-(c + r) // 256) for c, r in lanes]
    table = rng.permutation(sum(counts))
    kv = ops.KvPages(backend, K, D, len(table), table)
    pages = synthetic.kv_pages(rng, K, D, len(table)).reshape(len(table), -1)
    if case == "three rows":      # scales that are not finite, in slots past the sequences' ends alone, weigh nothing
        pages.view(np.uint16).reshape(len(table), -1)[table[counts[0] - 1], K * 256 * D + 256 - 8:K * 256 * D + 256] = 0x7E00
    kv.upload(pages)
    queries = rng.standard_normal((len(lanes), Q, 16, D)).astype(np.float16)
    tree = backend.from_array(_tree(rng, [r for _, r in lanes]))
    held = dict(kv=kv, first=np.concatenate([[0], np.cumsum(counts)])[:-1].tolist(), queries=backend.from_array(queries),
                sums=backend.from_array(queries.astype(np.float32).sum(-1)))
    most = max(r for _, r in lanes)
    tiles = max(1, (1 << (most - 1).bit_length()) * G // 16)
    for steps in (1, 4, 7):
        want = _partials(backend, f"attention_q8_split_d{D}_g{G}", 1, 256, heads, lanes, tree, held, steps)
        for t in (1, 2):
            kernel = f"attention_q8_few_d{D}_g{G}_t{t}"
            if t > tiles or not splash_amd.lib.sp_kernel_exists(kernel.encode()):
                continue
            print(f"case few {kernel} x {tiles // t} {case} steps {steps}", flush=True)
            got = _partials(backend, kernel, tiles // t, 64, heads, lanes, tree, held, steps)
            for lane, (a, b) in enumerate(zip(got, want)):
                assert np.array_equal(a[1], b[1]), (kernel, lane, "sums")
                seen = b[1][..., :1] != 0xFF800000      # (a split without a visible token may hold anything)
                assert np.array_equal(np.where(seen, a[0], 0), np.where(seen, b[0], 0)), (kernel, lane)


@pytest.mark.parametrize("rows,sequences,int8,kernel", [(1, 1, False, "few_d128_g8_t1"), (3, 1, False, "few_d128_g8_t1"),
                                                       (5, 1, False, "few_d128_g8_t1"), (8, 8, False, "few_d128_g8_t1"),
                                                       (9, 1, False, "split_d128_g8"), (1, 1, True, "q8q_split")])
def test_the_rule_takes_blocks_of_up_to_eight_rows(backend, rows, sequences, int8, kernel):
    plan = ops.AttentionPlan(64, 8, 128, [(i * rows, rows, 500, 2 * i) for i in range(sequences)], int8_queries=int8)
    kv = ops.KvPages(backend, 8, 128, 2 * sequences, np.arange(2 * sequences))
    graph = splash_amd.CommandGraph()
    n = rows * sequences
    ops.PagedAttention.add_attention(graph, plan, ops.AttentionWorkspace(backend, plan), backend.from_array(ops.chain_tree_rows([rows] * sequences)), kv,
                                     backend.allocate_buffer(n * 64 * 128 * 2))
    assert kernel in graph.kernels()[0], graph.kernels()
    backend.run(graph)


@pytest.mark.parametrize("heads,rows,tiles", [((64, 8, 128), 3, 2), ((64, 8, 128), 8, 4), ((32, 8, 128), 5, 2)])
def test_two_tiles_a_wave_once_the_parts_outnumber_the_simds(backend, heads, rows, tiles):
    """A tile a wave while every part has one of the device's SIMDs, four a compute unit, then two: the same rows, bit for bit."""
    print(f"case few parts {heads} rows={rows}", flush=True)
    Q, K, D = heads
    rng = np.random.default_rng(rows)
    lanes = [(0, rows, 700, 0), (rows, 2, 129, 3)]
    kv = ops.KvPages(backend, K, D, 4, rng.permutation(4))
    kv.upload(synthetic.kv_pages(rng, K, D, 4).reshape(4, -1))
    tree = backend.from_array(_tree(rng, [rows, 2]))
    queries = rng.standard_normal((2, Q, 16, D)).astype(np.float16)
    splits = ops.AttentionPlan(Q, K, D, lanes).splits
    enough = K * splits * len(lanes) * tiles // 4
    got = []
    for units, kernel in ((enough, "t1"), (enough - 1, "t2"), (1, "t2")):
        plan = ops.AttentionPlan(Q, K, D, lanes, compute_units=units)
        workspace = ops.AttentionWorkspace(backend, plan)
        workspace.queries.upload(queries)
        workspace.query_sums.upload(queries.astype(np.float32).sum(-1))
        graph, out = splash_amd.CommandGraph(), backend.from_array(np.full((rows + 2) * Q * D, 0x7FC0, np.uint16))
        ops.PagedAttention.add_attention(graph, plan, workspace, tree, kv, out)
        assert graph.kernels()[0].endswith(kernel), (units, graph.kernels())
        backend.run(graph)
        got.append(out.download(np.uint16))
    assert np.isfinite(orc.bf16_to_f32(got[0])).all() and all(np.array_equal(got[0], g) for g in got[1:])
    with pytest.raises(ValueError):
        ops.AttentionPlan(Q, K, D, lanes, compute_units=0)
