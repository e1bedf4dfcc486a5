"""GPU tests of a prompt chunk through the wide kernels (gguf_wide_*; model::DenseVerify::encodeWideChunkLayer): models of
2048 columns and more, chunks of more than 64 rows."""
import numpy as np
import pytest

from splash_amd import ops, synthetic, verify
from tests import oracle as orc
from tests.dense_reference import DenseModel

pytestmark = pytest.mark.gpu


def relative(a, b):
    a, b = orc.bf16_to_f32(a).astype(np.float64), orc.bf16_to_f32(b).astype(np.float64)
    return float(np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum()))


@pytest.mark.parametrize("down_format", [orc.FMT_Q4K, orc.FMT_Q5K, orc.FMT_Q6K])
@pytest.mark.parametrize("tokens", [65, 100, 129, 300])
def test_a_wide_chunk_is_its_blocks_to_rounding(backend, tokens, down_format):
    """Row counts that fill no, one and several 128-row workgroups and end inside a 16-row tile, an FFN width of nine
    super-blocks (half a piece of the table's pass), every format the kernels take: the hidden rows and the packed q|k|v
    rows of the last layer are those of the same blocks run sixteen rows a step, to the rounding of bf16 rows; under the
    staged rule to that of its half weights. A re-run repeats the bits."""
    print(f"case wide chunk tokens={tokens} down={down_format}", flush=True)
    H, layers = 2048, 1
    model = DenseModel(seed=31, hidden=H, q_heads=16, kv_heads=4, head_dim=128, ffn=2304, vocabulary=512, layers=layers,
                       down_format=orc.FMT_Q6K if down_format == orc.FMT_Q6K else orc.FMT_Q4K)
    if down_format == orc.FMT_Q5K:      # (the oracle quantizes to Q4_K and Q6_K)
        model.down_format, model.layers[0]["down"] = down_format, orc.make_native(down_format, H, 2304, 5)
    rng = np.random.default_rng(tokens)
    gpu = model.build_gpu(backend, max_lanes=1, context_tokens=[tokens + 300], prefill_rows=tokens)
    model.seed_context(gpu, None, rng)
    first, committed = model.table_first[0], 250
    prompt = rng.integers(0, 512, tokens).astype(np.uint32)
    pools = lambda: np.concatenate([gpu.buffer(verify.KV_POOL, layer).download(np.uint8) for layer in range(layers)])
    start = pools()
    rows_of = lambda which, rows, width: gpu.buffer(which, 0).download(np.uint16, rows * width).copy()
    hidden, qkv = [], []
    for at in range(0, tokens, 16):
        rows = min(16, tokens - at)
        lane = verify.Lane(rows, committed + at, table_first=first)
        gpu.set_block([lane], prompt[at:at + rows])
        backend.run(gpu.encode([lane], commit=False))
        hidden.append(rows_of(verify.HIDDEN, rows, H))
        qkv.append(rows_of(verify.QKV_ROWS, rows, 24 * 128))
    want_hidden, want_qkv = np.concatenate(hidden), np.concatenate(qkv)
    for staged in (False, True):
        gpu.set_staged_prefill(staged)
        seen = []
        for _ in range(2):
            for layer in range(layers):
                gpu.buffer(verify.KV_POOL, layer).upload(start.reshape(layers, -1)[layer])
            graph = gpu.encode_prefill(first, committed, tokens)
            assert any(name.startswith("gguf_wide_staged" if staged else "gguf_wide_q") for name in graph.kernels())
            gpu.set_prefill_block(prompt)
            backend.run(graph)
            seen.append((rows_of(verify.HIDDEN, tokens, H), rows_of(verify.QKV_ROWS, tokens, 24 * 128), pools()))
        assert all(np.array_equal(a, b) for a, b in zip(*seen))
        far = relative(seen[0][0], want_hidden), relative(seen[0][1], want_qkv)
        print(f"  staged={staged}: hidden {far[0]:.5f}, q|k|v {far[1]:.5f}", flush=True)
        # the q|k|v rows come of the same bf16 rows either way; the hidden rows of several bf16 roundings after them
        assert far[0] <= 9e-3 and far[1] <= (2.5e-3 if staged else 1e-3)


@pytest.mark.parametrize("tokens,experts,dense_ffn", [(257, 16, 0), (300, 80, 0), (300, 0, 512)])
def test_a_wide_hybrid_chunk_is_its_short_chunks_to_rounding(backend, tokens, experts, dense_ffn):
    """HybridVerify::encodeWidePrefillLayer: the experts' tasks (few and many rows an expert, a shared expert that every row
    visits, experts with no row), a packed width that ends inside a column group, an attention layer with gates, a dense
    FFN: the hidden rows and the recurrent state are those of the same prompt in chunks of 64 rows, which take the step's
    kernels, but for rows whose near-equal router scores rank the other way."""
    from tests.hybrid_reference import HybridModel
    print(f"case wide hybrid chunk tokens={tokens} experts={experts}", flush=True)
    H, V = 2048, 512
    model = HybridModel(seed=53, hidden=H, vocabulary=V, layers=4, q_heads=8, kv_heads=2, head_dim=128, gdn_key_heads=2, gdn_value_heads=4,
                        experts=experts, top_k=2 if experts else 0, expert_ffn=256 if experts else 0, shared_slices=1 if experts else 0,
                        shared_gate=bool(experts), gated_attention=True, dense_ffn=dense_ffn)
    gpu = model.build_gpu(backend, max_lanes=1, pages_per_lane=3, prefill_rows=tokens)
    rng = np.random.default_rng(tokens)
    model.seed_context(rng)
    model.seed_states(rng, lanes=1)
    committed = 200
    prompt = rng.integers(0, V, tokens).astype(np.uint32)
    start_pool, start_cells = gpu.buffer(verify.KV_POOL, 0).download(np.uint8), gpu.buffer(verify.GDN_STATES).download(np.uint8)

    def restore():
        gpu.buffer(verify.KV_POOL, 0).upload(start_pool)
        gpu.buffer(verify.GDN_STATES).upload(start_cells)

    def state(parity):
        cell = gpu.buffer(verify.GDN_STATES).download(np.uint8, gpu.cell_bytes, gpu.cell_offset(0, parity))
        return cell[gpu.strides.convolution_state_bytes:].view(np.float32).astype(np.float64)
    hidden, parity = [], 0
    restore()
    for at in range(0, tokens, 64):
        rows = min(64, tokens - at)
        gpu.set_prefill_block(prompt[at:at + rows])
        graph = gpu.encode_prefill(0, 0, committed + at, rows, parity=parity)
        assert not any("wide" in name for name in graph.kernels())
        backend.run(graph)
        hidden.append(gpu.buffer(verify.HIDDEN, 0).download(np.uint16, rows * H).copy())
        parity ^= 1
    want, want_state = orc.bf16_to_f32(np.concatenate(hidden)).reshape(tokens, H).astype(np.float64), state(parity)
    seen = []
    for _ in range(2):
        restore()
        gpu.set_prefill_block(prompt)
        graph = gpu.encode_prefill(0, 0, committed, tokens, parity=0)
        assert any("wide" in name for name in graph.kernels())
        backend.run(graph)
        seen.append((gpu.buffer(verify.HIDDEN, 0).download(np.uint16, tokens * H).copy(), state(1)))
    assert np.array_equal(seen[0][0], seen[1][0]) and np.array_equal(seen[0][1], seen[1][1])
    got = orc.bf16_to_f32(seen[0][0]).reshape(tokens, H).astype(np.float64)
    far = np.sqrt(((got - want) ** 2).sum(axis=1) / (want ** 2).sum(axis=1))
    far_state = np.sqrt(((seen[0][1] - want_state) ** 2).sum() / (want_state ** 2).sum())
    print(f"  rows: median {np.median(far):.5f}, 95th {np.percentile(far, 95):.5f}, worst {far.max():.5f}; state {far_state:.5f}", flush=True)
    assert np.median(far) <= 1e-2 and np.percentile(far, 90) <= 2e-2 and far_state <= 2e-2


@pytest.mark.parametrize("tokens", [511, 512, 525])
def test_chunks_of_many_blocks_prepare_a_block_a_workgroup(backend, tokens):
    """From 32 blocks on a chunk's head norms, RoPE and cache store take a workgroup a block (attention_q8_qkv_rows), a ragged
    last block among them, for plain heads and for gated ones with partial RoPE: held to the same bounds against the
    sixteen-row steps and the short chunks, whose workgroups take a row."""
    test_a_wide_chunk_is_its_blocks_to_rounding(backend, tokens, orc.FMT_Q4K)
    test_a_wide_hybrid_chunk_is_its_short_chunks_to_rounding(backend, tokens, 0, 512)


@pytest.mark.parametrize("tokens", [65, 300])
def test_an_exact_wide_model_chunk_equals_its_blocks(backend, tokens):
    """DenseVerify::setExactPrefill: a chunk that would take the wide kernels leaves the pages and the hidden rows of its
    blocks run as steps, bit for bit, whole or cut in two; the switch off, the wide kernels run again."""
    print(f"case exact chunk tokens={tokens}", flush=True)
    H, layers = 2048, 2
    model = DenseModel(seed=37, hidden=H, q_heads=16, kv_heads=4, head_dim=128, ffn=2304, vocabulary=512, layers=layers)
    rng = np.random.default_rng(tokens)
    gpu = model.build_gpu(backend, max_lanes=1, context_tokens=[tokens + 300], prefill_rows=tokens)
    model.seed_context(gpu, None, rng)
    first, committed = model.table_first[0], 250
    prompt = rng.integers(0, 512, tokens).astype(np.uint32)
    pools = lambda: np.concatenate([gpu.buffer(verify.KV_POOL, layer).download(np.uint8) for layer in range(layers)])
    rows_of = lambda rows: gpu.buffer(verify.HIDDEN, 0).download(np.uint16, rows * H).copy()
    start = pools()

    def restore():
        for layer in range(layers):
            gpu.buffer(verify.KV_POOL, layer).upload(start.reshape(layers, -1)[layer])
    hidden = []
    for at in range(0, tokens, 16):
        rows = min(16, tokens - at)
        lane = verify.Lane(rows, committed + at, table_first=first)
        gpu.set_block([lane], prompt[at:at + rows])
        backend.run(gpu.encode([lane], commit=False))
        hidden.append(rows_of(rows))
    want_hidden, want_pools = np.concatenate(hidden), pools()
    gpu.set_exact_prefill(True)
    for cuts in ([0, tokens], [0, 23, tokens]):
        restore()
        got = []
        for a, b in zip(cuts, cuts[1:]):
            gpu.set_prefill_block(prompt[a:b])
            graph = gpu.encode_prefill(first, committed + a, b - a)
            assert not any("wide" in name for name in graph.kernels())
            backend.run(graph)
            got.append(rows_of(b - a))
        assert np.array_equal(np.concatenate(got), want_hidden) and np.array_equal(pools(), want_pools)
    gpu.set_exact_prefill(False)
    assert any("wide" in name for name in gpu.encode_prefill(first, committed, tokens).kernels())


def test_an_exact_wide_hybrid_chunk_is_the_same_however_it_is_cut(backend):
    """HybridVerify::setExactPrefill: the chunk whole leaves the hidden rows, pages and recurrent state of the same prompt in
    chunks of 64 rows, bit for bit."""
    from tests.hybrid_reference import HybridModel
    print("case exact hybrid chunk", flush=True)
    H, V, tokens, committed = 2048, 512, 300, 200
    model = HybridModel(seed=59, hidden=H, vocabulary=V, layers=4, q_heads=8, kv_heads=2, head_dim=128, gdn_key_heads=2, gdn_value_heads=4,
                        experts=16, top_k=2, expert_ffn=256, shared_slices=1, shared_gate=True, gated_attention=True)
    gpu = model.build_gpu(backend, max_lanes=1, pages_per_lane=3, prefill_rows=tokens)
    rng = np.random.default_rng(tokens)
    model.seed_context(rng)
    model.seed_states(rng, lanes=1)
    prompt = rng.integers(0, V, tokens).astype(np.uint32)
    start_pool, start_cells = gpu.buffer(verify.KV_POOL, 0).download(np.uint8), gpu.buffer(verify.GDN_STATES).download(np.uint8)
    seen = []
    for size in (64, tokens):
        gpu.buffer(verify.KV_POOL, 0).upload(start_pool)
        gpu.buffer(verify.GDN_STATES).upload(start_cells)
        gpu.set_exact_prefill(size == tokens)
        hidden, parity = [], 0
        for at in range(0, tokens, size):
            rows = min(size, tokens - at)
            gpu.set_prefill_block(prompt[at:at + rows])
            graph = gpu.encode_prefill(0, 0, committed + at, rows, parity=parity)
            assert not any("wide" in name for name in graph.kernels())
            backend.run(graph)
            hidden.append(gpu.buffer(verify.HIDDEN, 0).download(np.uint16, rows * H).copy())
            parity ^= 1
        cell = gpu.buffer(verify.GDN_STATES).download(np.uint8, gpu.cell_bytes, gpu.cell_offset(0, parity))
        seen.append((np.concatenate(hidden), gpu.buffer(verify.KV_POOL, 0).download(np.uint8), cell))
    for got, want in zip(seen[1], seen[0]):
        assert np.array_equal(got, want)
    gpu.set_exact_prefill(False)
    assert any("wide" in name for name in gpu.encode_prefill(0, 0, committed, tokens).kernels())


@pytest.mark.parametrize("hidden,tokens", [(1024, 100), (2048, 40)])
def test_a_staged_chunk_allocates_nothing(backend, hidden, tokens):
    """The rows of the prefill tile are there once setStagedPrefill returns, also those of a model whose longer chunks take
    the wide kernels: encoding a chunk takes no memory, and cannot run out of it after dispatches were added to the graph."""
    print(f"case staged chunk memory hidden={hidden}", flush=True)
    model = DenseModel(seed=41, hidden=hidden, q_heads=16, kv_heads=4, head_dim=128, ffn=1024, vocabulary=512, layers=1)
    gpu = model.build_gpu(backend, max_lanes=1, context_tokens=[256], prefill_rows=128)
    before = backend.memory_stats().allocated_bytes
    gpu.set_staged_prefill(True)
    held = backend.memory_stats().allocated_bytes
    assert held - before >= 3 * 128 * 1024 * 2
    graph = gpu.encode_prefill(0, 0, tokens)
    assert any(name.startswith("gguf_prefill") for name in graph.kernels())
    assert backend.memory_stats().allocated_bytes == held


@pytest.mark.parametrize("values,exact", [(orc.FMT_Q4K, False), (orc.FMT_Q4K, True), (orc.FMT_Q6K, False)])
def test_only_a_driver_that_takes_the_wide_kernels_holds_their_buffers(backend, values, exact):
    """The wide kernels' table, SwiGLU rows and partials come with the last layer's weights, if all are tensors those kernels
    take (not with values of another format than the queries and keys) and chunks are not exact; encoding allocates nothing."""
    print(f"case wide memory values={values} exact={exact}", flush=True)
    H, F, rows = 2048, 2304, 300
    native = lambda n, k, fmt=orc.FMT_Q4K: (fmt, n, orc.make_native(fmt, n, k, n + k))
    project = lambda segments, k: ops.Projection.from_native(backend, segments, k)
    norm = lambda n: backend.from_array(orc.f32_to_bf16(np.ones(n, np.float32)))
    layer = (project([native(2048, H), native(512, H), native(512, H, values)], H), project([native(H, 2048)], 2048), project([native(F, H)], H),
             project([native(F, H)], H), project([native(H, F)], F), norm(H), norm(H), norm(128), norm(128))
    embedding, head = backend.from_array(native(512, H)[2]), ops.Projection.from_native(backend, [native(512, H)], H, float32=True)
    gpu = verify.DenseVerify(backend, H, 16, 4, 128, F, 512, 2, physical_pages=3, page_table_entries=2, prefill_rows=rows)
    gpu.set_exact_prefill(exact)
    held = lambda: backend.memory_stats().allocated_bytes
    created = held()
    gpu.set_layer(0, *layer)
    assert held() == created
    gpu.set_layer(1, *layer)
    gpu.set_head(orc.FMT_Q4K, embedding, norm(H), head)
    complete, wide = held(), values == orc.FMT_Q4K and not exact
    assert complete - created > rows * F * 2 if wide else complete - created < 1 << 16
    assert any("wide" in name for name in gpu.encode_prefill(0, 0, rows).kernels()) == wide
    assert held() == complete
    if exact:
        gpu.set_exact_prefill(False)
        switched = held()
        assert switched > complete and any("wide" in name for name in gpu.encode_prefill(0, 0, rows).kernels()) and held() == switched


@pytest.mark.parametrize("tokens", [40, 100])
def test_a_staged_chunk_refuses_ragged_tensors_whichever_kernels_take_it(backend, tokens):
    """Tensors that end inside a 128-column workgroup: the prefill tile refuses them, and so does a chunk of the same driver
    that is long enough for the wide kernels; without the staged rule both run."""
    print(f"case staged ragged tokens={tokens}", flush=True)
    H, F = 2048, 2304
    native = lambda n, k: (orc.FMT_Q4K, n, orc.make_native(orc.FMT_Q4K, n, k, n + k))
    project = lambda segments, k: ops.Projection.from_native(backend, segments, k)
    norm = lambda n: backend.from_array(orc.f32_to_bf16(np.ones(n, np.float32)))
    gpu = verify.DenseVerify(backend, H, 16, 4, 128, F, 512, 1, physical_pages=3, page_table_entries=2, prefill_rows=128)
    gpu.set_layer(0, project([native(1040, H), native(1008, H), native(1024, H)], H), project([native(H, 2048)], 2048), project([native(F, H)], H),
                  project([native(F, H)], H), project([native(H, F)], F), norm(H), norm(H), norm(128), norm(128))
    gpu.set_head(orc.FMT_Q4K, backend.from_array(native(512, H)[2]), norm(H), ops.Projection.from_native(backend, [native(512, H)], H, float32=True))
    assert len(gpu.encode_prefill(0, 0, tokens)) > 0
    gpu.set_staged_prefill(True)
    with pytest.raises(ValueError, match="128-column"):
        gpu.encode_prefill(0, 0, tokens)


def test_a_chunk_behind_millions_of_tokens_runs_in_windows(backend):
    """A history of more steps than a split counts: the whole-history attention cannot take it, the chunked one does. (The
    chunk is encoded, not run: its pages are named, not there.)"""
    print("case long history", flush=True)
    H, F, rows, limit = 2048, 256, 2048, 0xFFFF * 64
    native = lambda n, k: (orc.FMT_Q4K, n, orc.make_native(orc.FMT_Q4K, n, k, n + k))
    project = lambda segments, k: ops.Projection.from_native(backend, segments, k)
    norm = lambda n: backend.from_array(orc.f32_to_bf16(np.ones(n, np.float32)))
    gpu = verify.DenseVerify(backend, H, 16, 4, 128, F, 512, 1, physical_pages=2, page_table_entries=(limit >> 8) + 9, prefill_rows=rows)
    gpu.set_layer(0, project([native(2048, H), native(512, H), native(512, H)], H), project([native(H, 2048)], 2048), project([native(F, H)], H),
                  project([native(F, H)], H), project([native(H, F)], F), norm(H), norm(H), norm(128), norm(128))
    gpu.set_head(orc.FMT_Q4K, backend.from_array(native(512, H)[2]), norm(H), ops.Projection.from_native(backend, [native(512, H)], H, float32=True))
    for committed, wide in ((limit - rows, True), (limit - rows + 1, False)):
        assert any("wide" in name for name in gpu.encode_prefill(0, committed, rows).kernels()) == wide


_stage_model = {}


def stage_model(down):
    """The model of the stage tests with its down projection in a format."""
    H, F = 2048, 8448
    if not _stage_model:
        _stage_model["model"] = DenseModel(seed=61, hidden=H, q_heads=16, kv_heads=4, head_dim=128, ffn=F, vocabulary=512, layers=1, down_format=orc.FMT_Q6K)
        _stage_model[orc.FMT_Q6K] = _stage_model["model"].layers[0]["down"]
        _stage_model[orc.FMT_Q4K] = orc.quantize_rows(orc.FMT_Q4K, (np.random.default_rng(62).standard_normal((H, F), dtype=np.float32) * np.float32(0.02)))
        # Q5_K blocks of model-like scales: Q4_K's, the fifth bits drawn and the minimum's scale doubled
        drawn = np.random.default_rng(63)
        four = synthetic.q4k_native(drawn, H, F).reshape(-1, 144)
        four[:, 2:4] = (2 * four[:, 0:2].copy().view(np.float16)).view(np.uint8)
        fifth = drawn.integers(0, 256, (four.shape[0], 32), dtype=np.uint8)
        _stage_model[orc.FMT_Q5K] = np.ascontiguousarray(np.concatenate([four[:, :16], fifth, four[:, 16:]], axis=1)).ravel()
    model = _stage_model["model"]
    model.down_format, model.layers[0]["down"] = down, _stage_model[down]
    return model


@pytest.mark.parametrize("tokens,down,heights", [(100, orc.FMT_Q5K, ("_t4_g", "_t4_p")), (513, orc.FMT_Q6K, ("q4k_t6_g", "q6k_t7_p")),
                                                 (1300, orc.FMT_Q4K, ("q4k_t8_g", "q4k_t6_p")), (1543, orc.FMT_Q5K, ("q4k_t6_a", "q4k_t7_g", "q5k_t7_p"))])
def test_a_wide_chunks_stages_are_as_close_to_64_bits_as_the_steps(backend, tokens, down, heights):
    """Chunks whose plans take every tile height, K whole and in parts, an FFN wider than a table pass holds in one sweep, and
    (1543 rows) whole-history attention: each stage of the layer against 64-bit arithmetic on its own input rows, a row of
    every tile and all of the last ones, no further from it than the exact chunk's, on the whole and at the worst row."""
    print(f"case wide stages tokens={tokens} down={down}", flush=True)
    model = stage_model(down)
    d, w = model.dims, model.layers[0]
    H, F, W = d["hidden"], d["ffn"], 24 * 128
    rng = np.random.default_rng(tokens)
    gpu = model.build_gpu(backend, max_lanes=1, context_tokens=[tokens + 300], prefill_rows=tokens)
    model.seed_context(gpu, None, rng)
    prompt = rng.integers(0, 512, tokens).astype(np.uint32)
    picked = np.unique(np.concatenate([np.minimum(16 * np.arange((tokens + 15) // 16) + 7 * np.arange((tokens + 15) // 16) % 16, tokens - 1),
                                       np.arange(max(0, tokens - 20), tokens)]))
    wide64 = lambda bits: orc.bf16_to_f32(bits).astype(np.float64)
    weights = {name: orc.dequant_rows(down if name == "down" else orc.FMT_Q4K, w[name], n, k).astype(np.float64)
               for name, n, k in (("q", 2048, H), ("k", 512, H), ("v", 512, H), ("o", H, 2048), ("gate", F, H), ("up", F, H), ("down", H, F))}
    norm64 = lambda x, weight: x / np.sqrt((x * x).mean(axis=1, keepdims=True) + 1e-6) * wide64(weight)
    embedded = wide64(model.oracle_embedding(prompt))[picked]
    distance = {}
    for exact in (True, False):
        gpu.set_exact_prefill(exact)
        graph = gpu.encode_prefill(model.table_first[0], 250, tokens)
        names = graph.kernels()
        assert exact or all(any(name.startswith("gguf_wide_q") and height in name for name in names) for height in heights), names
        assert exact or tokens < 1543 or any("attention_q8_whole" in name for name in names)
        gpu.set_prefill_block(prompt)
        backend.run(graph)
        rows = lambda which, index, width: wide64(gpu.buffer(which, index).download(np.uint16, tokens * width).reshape(tokens, width)[picked])
        qkv, attention, middle, out = rows(verify.QKV_ROWS, 0, W), rows(verify.ATTENTION_ROWS, 0, 2048), rows(verify.HIDDEN, 1, H), rows(verify.HIDDEN, 0, H)
        n = norm64(embedded, w["input_norm"])
        m = norm64(middle, w["post_norm"])
        gate = m @ weights["gate"].T
        want = {"q|k|v": (qkv, np.concatenate([n @ weights[part].T for part in "qkv"], axis=1)),
                "output": (middle, embedded + attention @ weights["o"].T),
                "FFN": (out, middle + (gate / (1 + np.exp(-gate)) * (m @ weights["up"].T)) @ weights["down"].T)}
        for stage, (got, reference) in want.items():
            far = ((got - reference) ** 2).mean(axis=1) / (reference ** 2).mean(axis=1)
            distance[stage, exact] = np.sqrt(far.mean()), np.sqrt(far.max())
    for stage in ("q|k|v", "output", "FFN"):
        (a, worst_a), (b, worst_b) = distance[stage, True], distance[stage, False]
        print(f"  {stage}: exact {a:.3e} (worst row {worst_a:.3e}), wide {b:.3e} ({worst_b:.3e})", flush=True)
        # (an exact chunk rounds a norm's rows before their scale, a wide one after it: one rounding each, whose errors over
        # these rows differ by the draw, 0.3 % on the whole in exact arithmetic and 10 % at the worst row)
        assert b <= 1.03 * a and worst_b <= 1.5 * worst_a, stage


@pytest.mark.parametrize("tokens,experts,q_heads,kv_heads", [(300, 80, 8, 2), (300, 16, 8, 2), (784, 0, 32, 8)])
def test_a_wide_hybrid_chunk_layer_by_layer(backend, tokens, experts, q_heads, kv_heads):
    """HybridVerify::encodeWidePrefillLayer against the oracle from the GPU's own layer input, every row: a mixture whose
    routes take two windows, with a shared expert, a few tiles an expert and (16 experts) tasks of the tallest; gated attention over whole histories (784 rows of eight KV heads)."""
    from tests.hybrid_reference import HybridModel
    from tests.test_hybrid_step_gpu import close_bf16, sure_routes, ulps
    print(f"case wide hybrid layers tokens={tokens} experts={experts}", flush=True)
    H, V, committed = 2048, 512, 200
    model = HybridModel(seed=67, hidden=H, vocabulary=V, layers=4, q_heads=q_heads, kv_heads=kv_heads, head_dim=128, gdn_key_heads=2, gdn_value_heads=4,
                        experts=experts, top_k=8 if experts else 0, expert_ffn=256 if experts else 0, shared_slices=1 if experts else 0,
                        shared_gate=bool(experts), gated_attention=True, dense_ffn=0 if experts else 512)
    gpu = model.build_gpu(backend, max_lanes=1, pages_per_lane=4, prefill_rows=tokens)
    rng = np.random.default_rng(tokens)
    model.seed_context(rng)
    model.seed_states(rng, lanes=1)
    prompt = rng.integers(0, V, tokens).astype(np.uint32)
    gpu.set_prefill_block(prompt)
    hidden_of = lambda i=0: gpu.buffer(verify.HIDDEN, i).download(np.uint16, tokens * H).reshape(tokens, H)
    before = model.oracle_embedding(prompt)
    for layer in range(4):
        g = gpu.mixer_index(layer)
        if layer:
            before = hidden_of()
        if not model.attends(layer):
            conv_in, state_in = model.read_cell(0, 0, g)
        graph = gpu.encode_prefill(0, 0, committed, tokens, parity=0, first_layer=layer, layer_count=1)
        names = graph.kernels()
        assert any("gguf_wide_moe" in name for name in names) == bool(experts) and any("gguf_wide_q" in name for name in names)
        assert sum("gguf_wide_moe" in name and "_t8_" in name for name in names) == (2 if experts == 16 else 0), names
        assert any("attention_q8_whole" in name for name in names) == (model.attends(layer) and tokens == 784)
        backend.run(graph)
        packed = model.oracle_mixer_input(before, layer)
        if model.attends(layer):
            mixed = model.oracle_attention_chunk(packed, layer, 0, committed)
        else:
            w = model.layers[layer]
            want = orc.gdn_prefill(model.gdn_shape, packed, w["conv_w"], w["a_scale"], w["dt_bias"], w["mixer_norm"], conv_in, state_in)
            mixed = want["hidden"]
            conv, state = model.read_cell(0, 1, g)
            ok, detail = close_bf16(conv, want["conv_out"])
            assert ok and (ulps(conv, want["conv_out"]) > 0).mean() < 0.01, (layer, detail)
            assert np.abs(state - want["state_out"]).max() <= 2e-3 * np.abs(want["state_out"]).max(), layer
        ok, detail = close_bf16(hidden_of(1), model.oracle_mixer_output(mixed, before, layer))
        print(f"  layer {layer} mixer {detail}", flush=True)
        assert ok, ("mixer", layer, detail)
        scores, want = model.oracle_ffn(hidden_of(1), layer)
        sure = sure_routes(scores, 8) if experts else np.ones(tokens, bool)
        assert sure.mean() >= 0.9
        ok, detail = close_bf16(hidden_of()[sure], want[sure])
        print(f"  layer {layer} ffn {detail}, sure {sure.mean():.3f}", flush=True)
        assert ok, ("ffn", layer, detail)


@pytest.mark.parametrize("experts", [16, 0])
def test_encoding_a_wide_hybrid_chunk_allocates_nothing(backend, experts):
    """The hybrid driver's wide buffers come with the last layer's weights (HybridVerify::prepareChunks)."""
    from tests.hybrid_reference import HybridModel
    print(f"case wide hybrid memory experts={experts}", flush=True)
    model = HybridModel(seed=71, hidden=2048, vocabulary=512, layers=4, q_heads=8, kv_heads=2, head_dim=128, gdn_key_heads=2, gdn_value_heads=4,
                        experts=experts, top_k=2 if experts else 0, expert_ffn=256 if experts else 0, dense_ffn=0 if experts else 512)
    gpu = model.build_gpu(backend, max_lanes=1, pages_per_lane=3, prefill_rows=300)
    held = backend.memory_stats().allocated_bytes
    for rows, wide in ((256, False), (300, True)):
        assert any("wide" in name for name in gpu.encode_prefill(0, 0, 0, rows).kernels()) == wide
        assert backend.memory_stats().allocated_bytes == held
