"""The passes that open and close a step as one dispatch each, bit for bit the separate ones."""
import ctypes

import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc

pytestmark = pytest.mark.gpu
U32, U64 = ctypes.c_uint32, ctypes.c_uint64


class Embed(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("rows", "vocabulary", "hidden", "tiles", "pairs", "rope_rows", "sequences", "reserved")] + [
        ("first_row", U32 * 8), ("row_count", U32 * 8), ("anchor", U32 * 8)]


# one super-block; a step's rows; a second row tile; the widest row a workgroup holds, without rotary pairs; more pairs than
# threads; a last wave half filled with vectors. By the threads that a step's entry has, and by 256.
@pytest.mark.parametrize("threads", ["the entry's", 256])
@pytest.mark.parametrize("rows,hidden,pairs", [(1, 256, 32), (16, 5120, 64), (17, 2304, 1), (33, 8192, 0), (5, 1024, 300), (3, 768, 64)])
@pytest.mark.parametrize("fmt", ops.FORMATS)
def test_gather_norm_and_rope_tables_in_one_pass(backend, fmt, rows, hidden, pairs, threads):
    threads = min(hidden, 1024) if threads != 256 else threads
    print(f"case entry fmt={fmt} rows={rows} hidden={hidden} pairs={pairs} threads={threads}", flush=True)
    vocabulary = 40
    rng = np.random.default_rng(rows)
    table = backend.from_array(orc.make_native(fmt, vocabulary, hidden, 3))
    ids = rng.integers(0, vocabulary, rows).astype(np.uint32)
    ids[-1] = vocabulary   # past the vocabulary: zeros
    tokens, weight = backend.from_array(ids), backend.from_array(orc.f32_to_bf16((1 + 0.2 * rng.standard_normal(hidden)).astype(np.float32)))
    cut = (rows + 1) // 2
    sequences = [(0, cut, 32752)] + ([(cut, rows - cut, 7)] if rows > cut else [])
    inverse = backend.from_array((1e6 ** (-np.arange(max(pairs, 1)) / max(pairs, 1))).astype(np.float32))
    depth = backend.from_array(rng.integers(0, 16, rows).astype(np.uint32))
    outputs = lambda: [backend.from_array(np.full(n, 0xA5, np.uint8)) for n in (rows * hidden * 2, rows * hidden * 2, ops.gguf_table_bytes(hidden, rows),
                                                                           max(rows * pairs, 1) * 4, max(rows * pairs, 1) * 4)]
    apart, together = outputs(), outputs()
    graph = splash_amd.CommandGraph()
    if pairs:
        ops.RoPE.add_tree_tables(graph, inverse, depth, apart[3], apart[4], pairs, sequences)
    ops.Embedding.add(graph, fmt, table, vocabulary, hidden, tokens, apart[0], rows)
    ops.Normalization.add_rms_table(graph, apart[0], weight, apart[1], apart[2], hidden, rows)
    name = graph.kernels()[-2]
    tiles = (rows + 15) // 16
    p = Embed(rows, vocabulary, hidden, tiles, pairs, rows, len(sequences), 0)
    for i, (first, count, anchor) in enumerate(sequences):
        p.first_row[i], p.row_count[i], p.anchor[i] = first, count, anchor
    graph.add(name.replace("gguf_embed_", "gguf_embed_norm_"), [table, tokens, weight, *together[:3], inverse, depth, *together[3:]], p,
              (tiles * 16, 2 if pairs else 1, 1), (threads, 1, 1))
    backend.run(graph)
    for a, b in zip(apart, together):
        assert np.array_equal(a.download(), b.download())


class Sequence(ctypes.Structure):
    _fields_ = [("first_row", U32), ("committed", U32), ("table_first", U32), ("rows", ctypes.c_uint16), ("steps_per_split", ctypes.c_uint16)]


class Commit(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("kv_heads", "head_dim", "sequences", "layers")] + [("page_bytes", U64), ("layer_bytes", U64), ("sequence", Sequence * 8)]


class AcceptCommit(ctypes.Structure):
    _fields_ = [("commit", Commit), ("remaining", U32 * 8), ("stop_tokens", U32 * 4)]


@pytest.mark.parametrize("dimension,kv_heads", [(64, 2), (128, 3)])
def test_selection_acceptance_and_commit_in_one_dispatch(backend, dimension, kv_heads):
    """Chains and trees of 1 to 16 rows, caps, stop tokens, paths across a page's end, rows with no selectable logit, lanes
    that keep no row."""
    from tests.test_oracle_sampling import random_tree
    from tests.test_glue_sampling_gpu import sampling_buffers
    rng = np.random.default_rng(dimension)
    layers, vocabulary = 2, 700
    page_bytes = 2 * kv_heads * 256 * dimension + 2 * kv_heads * 256 * 2
    for trial in range(12):
        print(f"case accept commit d={dimension} trial={trial}", flush=True)
        counts = [16, 1] if trial == 0 else [int(rng.integers(1, 17)) for _ in range(int(rng.integers(1, 9)))]
        first = np.concatenate([[0], np.cumsum(counts)])
        rows = int(first[-1])
        lanes = [(int(first[i]), n) for i, n in enumerate(counts)]
        tree = np.concatenate([random_tree(rng, n) if trial % 2 else ops.chain_tree_rows([n]) for n in counts])
        if trial > 8:   # a lane whose anchor is not its own ancestor keeps no row: its commit takes the rows left there before
            tree["ancestors"][first[int(rng.integers(0, len(counts)))]] = 0
        tokens = rng.integers(0, 3, rows).astype(np.uint32)
        logits = rng.standard_normal((rows, vocabulary)).astype(np.float32)
        logits[np.arange(rows), rng.integers(0, 3, rows)] = 9.0
        logits[rng.integers(0, rows)] = np.nan
        remaining = [int(rng.integers(1, 20)) for _ in counts]
        stops = (2, ops.NO_TOKEN, ops.NO_TOKEN, ops.NO_TOKEN) if trial % 3 == 0 else (ops.NO_TOKEN,) * 4
        p = AcceptCommit(Commit(kv_heads, dimension, len(counts), layers, page_bytes, 2 * len(counts) * page_bytes))
        for i, n in enumerate(counts):
            p.commit.sequence[i] = Sequence(int(first[i]), int(rng.integers(235, 256)), 2 * i, n, 1)
            p.remaining[i] = remaining[i]
        for i, s in enumerate(stops):
            p.stop_tokens[i] = s
        table = backend.from_array(rng.permutation(2 * len(counts)).astype(np.uint64))
        pool = rng.integers(0, 256, layers * 2 * len(counts) * page_bytes, dtype=np.uint8)
        before = [np.array([int(rng.integers(0, 1 << n)) for n in counts], np.uint32) for _ in range(3)]
        results = []
        for together in (False, True):
            b = sampling_buffers(backend, rows, vocabulary, logits, tokens=tokens, tree=tree)
            kv = backend.from_array(pool)
            left = [backend.from_array(x) for x in before]
            graph = splash_amd.CommandGraph()
            ops.Sampling.add_verify(graph, b, vocabulary, vocabulary, lanes, [0.0] * len(counts))
            if together:
                backend.run(graph)
                graph = splash_amd.CommandGraph()
                b["tokens"] = backend.from_array(np.full(rows, 0xA5, np.uint32))   # it reads the shards' partials alone
                graph.add("attention_q8_accept_commit_d%d" % dimension, [b["partial_values"], b["partial_indices"], b["input_tokens"], b["tree_rows"], b["tokens"],
                                                                        *left, table, kv], p, (kv_heads, len(counts), layers), (dimension, 1, 1))
            else:
                ops.Sampling.add_acceptance(graph, b["input_tokens"], b["tree_rows"], b["tokens"], *left, lanes, remaining, stops)
                graph.add("attention_q8_commit_d%d" % dimension, [left[2], table, kv], p.commit, (kv_heads, len(counts), layers), (dimension, 1, 1))
            backend.run(graph)
            results.append([b["tokens"].download(), *(x.download() for x in left), kv.download()])
        for a, b in zip(*results):
            assert np.array_equal(a, b)


# a workgroup's LDS holds a row's last column, the first row it does not hold, and a model without rotary pairs
@pytest.mark.parametrize("hidden,pairs,entry", [(8192, 32, ["gguf_embed_norm_q4k"]), (512, 0, ["gguf_embed_norm_q4k"]),
                                                (8448, 32, ["rope_build_tree_tables", "gguf_embed_q4k", "norm_rms_table16"]),
                                                (8448, 0, ["gguf_embed_q4k", "norm_rms_table16"])])
def test_a_steps_entry_takes_one_pass_where_a_row_fits(backend, hidden, pairs, entry):
    """The first layer's projection of a step's rows is, bit for bit, that of the embedding and the layer on their own."""
    print(f"case entry rule hidden={hidden} pairs={pairs}", flush=True)
    from splash_amd import verify
    from tests.dense_reference import DenseModel
    Q, K, D, ffn, vocabulary = 4, 2, 64, 256, 512
    m = DenseModel(3, hidden, Q, K, D, ffn, vocabulary, 1)
    gpu = verify.DenseVerify(backend, hidden, Q, K, D, ffn, vocabulary, 1, rotary_pairs=pairs, max_lanes=2, physical_pages=2)
    gpu.buffer(verify.PAGE_TABLE).upload(np.arange(2, dtype=np.uint64))
    P, w, f = ops.Projection.from_native, m.layers[0], orc.FMT_Q4K
    gpu.set_layer(0, P(backend, [(f, Q * D, w["q"]), (f, K * D, w["k"]), (f, K * D, w["v"])], hidden), P(backend, [(f, hidden, w["o"])], Q * D),
                  P(backend, [(f, ffn, w["gate"])], hidden), P(backend, [(f, ffn, w["up"])], hidden), P(backend, [(f, hidden, w["down"])], ffn),
                  *(backend.from_array(w[n]) for n in ("input_norm", "post_norm", "q_norm", "k_norm")))
    gpu.set_head(f, backend.from_array(m.embedding), backend.from_array(m.final_norm), P(backend, [(orc.FMT_Q6K, vocabulary, m.head)], hidden, float32=True))
    lanes = [verify.Lane(16, 0), verify.Lane(3, 0, table_first=1)]
    gpu.set_block(lanes, np.random.default_rng(1).integers(0, vocabulary + 1, 19).astype(np.uint32))
    got = []
    graph = gpu.encode(lanes, commit=False)
    assert graph.kernels()[:len(entry)] == entry, graph.kernels()
    for run in (graph, gpu.encode_part(1, 0, lanes, gpu.encode_part(0, 0, lanes))):
        for which in (verify.QKV_ROWS, verify.ATTENTION_ROWS):
            rows = gpu.buffer(which)
            rows.upload(np.full(rows.size_bytes // 2, 0x7FC0, np.uint16))
        backend.run(run)
        got.append([gpu.buffer(which).download(np.uint16) for which in (verify.QKV_ROWS, verify.ATTENTION_ROWS)])
    for whole, parts, width in zip(*got, ((Q + 2 * K) * D, Q * D)):
        assert np.isfinite(orc.bf16_to_f32(whole[:19 * width])).all() and np.array_equal(whole, parts)
