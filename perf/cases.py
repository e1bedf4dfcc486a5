"""What the framework's speed is measured on: the work a serving engine has this library do, through its Python entry points.

Every case is one call the engine makes between two looks at the request queue: a verify step of a dense or a hybrid
target (the block's rows written, the step encoded for the lanes as they stand, run, its results read: a lane's committed
length changes with every step, so the engine encodes each one), a prompt chunk through either target, the draft model's
forward pass, and the selection of the rows to verify from a draft's logits. The models are the shapes the benchmark names
(the 27B-shaped dense decoder, the 35B-A3B-shaped hybrid, the two-layer plumbing shape) with fewer of their layers: layers
are alike, so a layer's and the head's share of the time is what a deeper model's is, and the 16-bit roundings of few layers
stay small enough for two correct runs to be compared.

Weights are GGUF blocks with uniform codes and model-like scales, dealt at random from a packed pool into images of their
own for every layer. The layers add a little each to the residual stream, and the head partly agrees with the embedding of
the token before, so that logits have the margin a trained model's have and a drafted chain is accepted up to a point.
"""
import ctypes
import math

import numpy as np
import torch

import splash_amd
from splash_amd import ops, synthetic, verify

DENSE = {
    # the benchmark's 27B shape (64 such layers) and its plumbing shape
    "27b": dict(hidden=5120, q_heads=64, kv_heads=8, head_dim=128, ffn=25600, vocabulary=151936),
    "small": dict(hidden=1024, q_heads=16, kv_heads=8, head_dim=64, ffn=3072, vocabulary=32000),
}
# the benchmark's 35B-A3B shape (48 layers, every fourth attends)
HYBRID = dict(hidden=2048, q_heads=32, kv_heads=4, head_dim=128, gdn_key_heads=16, gdn_value_heads=32, experts=128, top_k=8,
              expert_ffn=768, vocabulary=151936)
# the benchmark's draft model at the 27B target's widths: five layers, the target's head
DRAFT = dict(hidden=5120, intermediate=13824, layers=5, target_layers=5, vocabulary=151936)
NEXT_TILES = 37          # the model continues token t with t + 16 * NEXT_TILES
POOL = 96                # distinct 16-column x 256-input records of a weight pool
PAGE = ops.PAGE_TOKENS
Q4, Q6 = 144 / 256, 210 / 256    # bytes a weight


def listed():
    return [
        # The smallest model a deployment runs, one request: launches and host work count.
        dict(name="dense small 1x16", kind="dense", model="small", layers=2, lanes=1, rows=16, context=512, ragged=False, temperature=0.0),
        # The headline step: one request, a 16-token draft block, 32K tokens of context.
        dict(name="dense 27b 1x16 32k", kind="dense", model="27b", layers=8, lanes=1, rows=16, context=32752, ragged=False, temperature=0.0),
        # Plain decoding of one request without a draft, at a long context.
        dict(name="dense 27b 1x1 100k", kind="dense", model="27b", layers=8, lanes=1, rows=1, context=100003, ragged=False, temperature=0.0),
        # Four requests at once, full blocks.
        dict(name="dense 27b 4x16 32k", kind="dense", model="27b", layers=8, lanes=4, rows=16, context=32752, ragged=False, temperature=0.0),
        # Requests of a chat service: blocks and contexts of different lengths, sampled.
        dict(name="dense 27b ragged sampled", kind="dense", model="27b", layers=8, lanes=3, rows=11, context=5003, ragged=True, temperature=0.7),
        # A long prompt's chunk after 8K tokens, and the odd tail of a short one, through the step's kernels (the default).
        dict(name="prefill 27b 2048", kind="prefill", model="27b", layers=4, tokens=2048, committed=8192, staged=False),
        dict(name="prefill 27b 777", kind="prefill", model="27b", layers=4, tokens=777, committed=0, staged=False),
        # A chunk with the prefill tile switched on.
        dict(name="prefill 27b staged 1536", kind="prefill", model="27b", layers=4, tokens=1536, committed=4096, staged=True),
        # The hybrid target's step: eight requests that each fold the rows kept of the step before; and its prompt chunk.
        dict(name="hybrid 35b 8x16 16k", kind="hybrid", layers=8, lanes=8, rows=16, context=16368, ragged=False),
        dict(name="hybrid prefill 35b 2048", kind="hybrid_prefill", layers=8, tokens=2048, committed=4096),
        # The draft model's forward pass for one request, and the selection of eight requests' rows.
        dict(name="draft 1", kind="draft", lanes=1, cached=40000),
        dict(name="select 8", kind="select", lanes=8, children=3),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "prefill", "prefill", "hybrid", "hybrid", "hybrid_prefill", "draft", "select"])
    if kind == "dense":
        model = rng.choice(["27b", "27b", "small"])
        lanes = rng.randint(1, 4)
        return dict(kind=kind, model=model, layers=8 if model == "27b" else 2, lanes=lanes, rows=rng.randint(1, 16),
                    context=_log(rng, 60, 100000 // lanes), ragged=rng.random() < 0.5, temperature=rng.choice([0.0, 0.0, 0.7]))
    if kind == "prefill":
        staged = rng.random() < 0.4
        return dict(kind=kind, model="27b", layers=4, tokens=_log(rng, 17, 1536 if staged else 2048), committed=rng.randint(0, 8192), staged=staged)
    if kind == "hybrid":
        return dict(kind=kind, layers=8, lanes=rng.randint(1, 8), rows=rng.randint(1, 16), context=_log(rng, 60, 16368), ragged=rng.random() < 0.5)
    if kind == "hybrid_prefill":
        return dict(kind=kind, layers=8, tokens=_log(rng, 17, 2048), committed=rng.randint(0, 4096))
    if kind == "draft":
        return dict(kind=kind, lanes=rng.randint(1, 8), cached=_log(rng, 20, 40000))
    return dict(kind=kind, lanes=rng.randint(1, 8), children=rng.randint(1, 4))


# ------------------------------------------------------------------------------------------------ device memory
_shared = {}


def _backend():
    """The process's one backend, as an engine holds it."""
    if "backend" not in _shared:
        torch.cuda.init()
        _shared["backend"] = splash_amd.Backend(0)
    return _shared["backend"]


class _Memory:
    """Bytes of a device buffer; a tensor over them keeps this object, and with it the buffer, alive."""

    def __init__(self, buffer, offset, count):
        if offset < 0 or count < 1 or offset + count > buffer.size_bytes:
            raise ValueError("bytes outside the buffer")
        self.buffer = buffer
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="|u1", data=(buffer.gpu_address + offset, False), version=2)


def _bytes(buffer, offset=0, count=None):
    """A device buffer's bytes as a torch tensor over the same memory."""
    count = buffer.size_bytes - offset if count is None else count
    return torch.as_tensor(_Memory(buffer, offset, count), device="cuda")


def _values(buffer, dtype, *shape):
    count = math.prod(shape) * dtype.itemsize
    return _bytes(buffer, 0, count).view(dtype).view(*shape)


def _strided(buffer, dtype, offset, shape, strides):
    """Values of `dtype` in a buffer: byte offset and byte strides."""
    size = dtype.itemsize
    flat = _bytes(buffer, 0, buffer.size_bytes // size * size).view(dtype)
    return flat.as_strided(shape, [s // size for s in strides], offset // size)


class _Maker:
    """Makes a state's device buffers from a seed."""

    def __init__(self, seed):
        self.backend = _backend()
        self.rng = np.random.default_rng(seed)
        self.torch = torch.Generator(device="cuda")
        self.torch.manual_seed(seed)
        self.pools = {}

    def pool(self, fmt, std):
        """POOL packed records of a format whose weights have this standard deviation."""
        if (fmt, std) not in self.pools:
            native = synthetic.native(self.rng, fmt, 16 * POOL, 256)
            _scale(fmt, native, std / 0.02)
            packed = ops.pack_gguf_image(fmt, native, 16 * POOL, 256)
            self.pools[fmt, std] = torch.from_numpy(packed).cuda().view(POOL, -1)
        return self.pools[fmt, std]

    def image(self, fmt, n, k, std=0.02, copies=1):
        """`copies` weight images of [n][k] one after the other in a buffer."""
        pool = self.pool(fmt, std)
        return self._dealt(pool, torch.randint(0, POOL, (copies * (n // 16) * (k // 256),), device="cuda", generator=self.torch))

    def _dealt(self, pool, index):
        out = self.backend.allocate_buffer(index.numel() * pool.shape[1], label="weights")
        torch.index_select(pool, 0, index.view(-1), out=_bytes(out).view(-1, pool.shape[1]))
        return out

    def projection(self, segments, k, std=0.02, float32=False):
        return ops.Projection([(fmt, n, self.image(fmt, n, k, std)) for fmt, n in segments], k, float32)

    def bf16(self, values):
        return self.backend.from_array((np.ascontiguousarray(values, np.float32).view(np.uint32) >> 16).astype(np.uint16))

    def norm(self, n, mean=1.0):
        return self.bf16(mean * (1 + 0.05 * self.rng.standard_normal(n)))

    def normal(self, buffer, dtype, count, std, offset=0):
        """Fills `count` values of a buffer with N(0, std)."""
        view = _bytes(buffer, offset, count * dtype.itemsize).view(dtype)
        for at in range(0, count, 1 << 26):
            part = view[at:at + (1 << 26)]
            part.copy_(torch.randn(part.shape, device="cuda", generator=self.torch) * std)

    def embedding_and_head(self, vocabulary, hidden):
        """The token table (native Q4_K rows, values near 1) and the Q6_K head, which over a part of its inputs holds the
        codes of the token NEXT_TILES column tiles before."""
        blocks, tiles = hidden // 256, vocabulary // 16
        agree = max(2, min(4, blocks // 2))
        native = synthetic.q4k_native(self.rng, 16 * POOL, 256)
        codes = _q4k_codes(native.reshape(-1, 144))
        head = ops.pack_gguf_image(ops.FMT_Q6K, _q6k_of_codes(self.rng, codes), 16 * POOL, 256)
        _scale(ops.FMT_Q4K, native, 50.0)
        rows = torch.from_numpy(native).cuda().view(POOL, 16, 144)
        index = torch.randint(0, POOL, (tiles, blocks), device="cuda", generator=self.torch)
        embedding = self.backend.allocate_buffer(vocabulary * blocks * 144, label="embedding")
        table = _bytes(embedding).view(tiles, 16, blocks, 144)
        for block in range(blocks):
            table[:, :, block] = rows[index[:, block]]
        other = torch.randint(0, POOL, (tiles, blocks), device="cuda", generator=self.torch)
        other[:, :agree] = index.roll(NEXT_TILES, 0)[:, :agree]
        image = self._dealt(torch.from_numpy(head).cuda().view(POOL, -1), other)
        return embedding, ops.Projection([(ops.FMT_Q6K, vocabulary, image)], hidden, float32=True)

    def kv_pool(self, buffer, layers, physical, kv_heads, head_dim):
        """Every layer's pages of an INT8 context, dealt from a few."""
        few = torch.from_numpy(synthetic.kv_pages(self.rng, kv_heads, head_dim, 3)).cuda()
        at = torch.randint(0, 3, (layers * physical,), device="cuda", generator=self.torch)
        torch.index_select(few, 0, at, out=_bytes(buffer).view(layers * physical, -1))

    def chain(self, rows, vocabulary):
        """A lane's block: an anchor and a draft whose first half is what the model says."""
        tokens = [int(self.rng.integers(0, vocabulary))]
        for row in range(1, rows):
            tokens.append((tokens[-1] + 16 * NEXT_TILES) % vocabulary if row <= rows // 2 else int(self.rng.integers(0, vocabulary)))
        return tokens


def _scale(fmt, native, factor):
    """Multiplies the blocks' fp16 scales in place."""
    at, size, count = (0, 144, 2) if fmt == ops.FMT_Q4K else (208, 210, 1)
    blocks = native.reshape(-1, size)
    d = np.ascontiguousarray(blocks[:, at:at + 2 * count]).view(np.float16).astype(np.float32) * factor
    blocks[:, at:at + 2 * count] = d.astype(np.float16).view(np.uint8)


def _q4k_codes(blocks):
    """The 256 4-bit codes of native Q4_K blocks, in input order."""
    q = blocks[:, 16:].reshape(-1, 4, 32)
    return np.stack([q & 15, q >> 4], axis=2).reshape(-1, 256)


def _q6k_of_codes(rng, codes):
    """Native Q6_K blocks whose values are proportional to code - 7.5, standard deviation near 0.02."""
    q = (2 * codes.astype(np.int32) + 17).astype(np.uint8).reshape(-1, 2, 4, 32)
    out = np.empty((q.shape[0], 210), np.uint8)
    low, high = q & 15, q >> 4
    out[:, :128] = np.stack([low[:, :, 0] | low[:, :, 2] << 4, low[:, :, 1] | low[:, :, 3] << 4], axis=2).reshape(-1, 128)
    out[:, 128:192] = (high[:, :, 0] | high[:, :, 1] << 2 | high[:, :, 2] << 4 | high[:, :, 3] << 6).reshape(-1, 64)
    out[:, 192:208] = rng.integers(30, 37, (q.shape[0], 16)).astype(np.uint8)
    out[:, 208:210] = np.full((q.shape[0], 1), 0.02 / 33 / 9.2, np.float16).view(np.uint8)
    return out.reshape(-1)


# ------------------------------------------------------------------------------------------------ targets
def _down_std(hidden, ffn):
    """A down projection that adds about 0.15 to a residual stream of size 1: SwiGLU rows are near 0.65 * (0.02^2 hidden)."""
    return round(0.15 / (math.sqrt(ffn) * 0.65 * 0.0004 * hidden), 6)


def _dense_target(make, case, physical, entries, lanes, prefill_rows):
    m = DENSE[case["model"]]
    H, D, F, V = m["hidden"], m["head_dim"], m["ffn"], m["vocabulary"]
    QW, KW = m["q_heads"] * D, m["kv_heads"] * D
    gpu = verify.DenseVerify(make.backend, H, m["q_heads"], m["kv_heads"], D, F, V, case["layers"], max_lanes=lanes, physical_pages=physical,
                             page_table_entries=entries, prefill_rows=prefill_rows)
    q4, q6 = ops.FMT_Q4K, ops.FMT_Q6K
    for layer in range(case["layers"]):
        gpu.set_layer(layer, make.projection([(q4, QW), (q4, KW), (q4, KW)], H), make.projection([(q4, H)], QW, 0.01), make.projection([(q4, F)], H),
                      make.projection([(q4, F)], H), make.projection([(q6, H)], F, _down_std(H, F)), make.norm(H), make.norm(H), make.norm(D, 2.0),
                      make.norm(D))
    embedding, head = make.embedding_and_head(V, H)
    gpu.set_head(q4, embedding, make.norm(H), head)
    make.kv_pool(gpu.buffer(verify.KV_POOL, 0), 1, physical, m["kv_heads"], D)
    first = _bytes(gpu.buffer(verify.KV_POOL, 0))
    for layer in range(1, case["layers"]):
        pages = _bytes(gpu.buffer(verify.KV_POOL, layer)).view(physical, -1)
        torch.index_select(first.view(physical, -1), 0, torch.randperm(physical, device="cuda", generator=make.torch), out=pages)
    return gpu


def _hybrid_target(make, case, physical, entries, lanes, prefill_rows):
    m = HYBRID
    H, D, V, E, F = m["hidden"], m["head_dim"], m["vocabulary"], m["experts"], m["expert_ffn"]
    gpu = verify.HybridVerify(make.backend, H, V, case["layers"], m["q_heads"], m["kv_heads"], D, m["gdn_key_heads"], m["gdn_value_heads"], E,
                              m["top_k"], F, max_lanes=lanes, physical_pages=physical, page_table_entries=entries, prefill_rows=prefill_rows)
    packed, QKV, QW, GW = gpu.dims.gdn_packed_width, (m["q_heads"] + 2 * m["kv_heads"]) * D, m["q_heads"] * D, m["gdn_value_heads"] * 128
    VH, conv = m["gdn_value_heads"], (2 * m["gdn_key_heads"] + m["gdn_value_heads"]) * 128
    q4, q6, rng = ops.FMT_Q4K, ops.FMT_Q6K, make.rng
    for layer in range(case["layers"]):
        experts = dict(router=make.projection([(q6, E)], H, 0.06, float32=True), gate_images=make.image(q4, F, H, copies=E),
                       up_images=make.image(q4, F, H, copies=E), down_images=make.image(q4, H, F, _down_std(H, F), copies=E))
        if gpu.attends(layer):
            mixer = (make.projection([(q4, QKV)], H), make.projection([(q4, H)], QW, 0.01))
            small = dict(query_norm=make.norm(D, 2.0), key_norm=make.norm(D))
        else:
            mixer = (make.projection([(q4, packed)], H), make.projection([(q4, H)], GW, 0.005))
            small = dict(convolution_weights=make.bf16(rng.standard_normal((conv, 4)) * 0.4),
                         decay_weights=make.backend.from_array((-np.exp(rng.uniform(-1, 1, VH))).astype(np.float32)),
                         time_bias=make.bf16(rng.uniform(-1, 1, VH)), mixer_norm=make.norm(128))
        gpu.set_layer(layer, *mixer, input_norm=make.norm(H), post_norm=make.norm(H), **experts, **small)
    embedding, head = make.embedding_and_head(V, H)
    gpu.set_head(q4, embedding, make.norm(H), head)
    for layer in range(case["layers"] // 4):
        make.kv_pool(gpu.buffer(verify.KV_POOL, layer), 1, physical, m["kv_heads"], D)
    states = gpu.buffer(verify.GDN_STATES)
    make.normal(states, torch.float32, states.size_bytes // 4, 0.05)
    for cell in range(2 * lanes):      # the carries are bf16 rows, before a cell's states
        make.normal(states, torch.bfloat16, gpu.strides.convolution_state_bytes // 2, 1.0, cell * gpu.cell_bytes)
    return gpu


def _lanes(case):
    """(rows, committed) of each lane: alike, or a full one and shorter ones."""
    if not case["ragged"]:
        return [(case["rows"], case["context"])] * case["lanes"]
    return [(max(1, case["rows"] - 3 * lane), max(0, case["context"] - 1237 * lane)) for lane in range(case["lanes"])]


def _tables(make, counts, written):
    """The page table of sequences of these many pages in random places, the last `written[i]` pages of each, which the
    call writes, side by side from page 0 on; returns it, the physical pages and every sequence's first entry."""
    table, first, at = [], [], 0
    free = sum(written) + make.rng.permutation(sum(counts) - sum(written))
    used = 0
    for count, tail in zip(counts, written):
        first.append(len(table))
        table += [int(p) for p in free[used:used + count - tail]] + list(range(at, at + tail))
        used, at = used + count - tail, at + tail
    return np.array(table, np.uint64), sum(counts), first


def _cached_scales(gpu, layers, pages, kv_heads, head_dim):
    """The fp16 scales of the first `pages` physical pages of every layer: [layers][pages][2][kv_heads][256]."""
    size, codes = gpu.physical_pages * _page_bytes(kv_heads, head_dim), 2 * kv_heads * PAGE * head_dim
    views = []
    for layer in range(layers):
        views.append(_strided(gpu.buffer(verify.KV_POOL, layer).view(0, size), torch.float16, codes, (pages, 2 * kv_heads * PAGE),
                              (_page_bytes(kv_heads, head_dim), 2)))
    return views


def _page_bytes(kv_heads, head_dim):
    return ops.kv_page_bytes(kv_heads, head_dim)


class _Step:
    """A verify step of a target's lanes."""

    def __init__(self, case, seed):
        make = _Maker(seed)
        hybrid = case["kind"] == "hybrid"
        m = HYBRID if hybrid else DENSE[case["model"]]
        V, H = m["vocabulary"], m["hidden"]
        shape = _lanes(case)
        counts = [max(2, -(-(committed + rows) // PAGE)) for rows, committed in shape]
        table, physical, first = _tables(make, counts, [2] * len(counts))
        self.gpu = gpu = (_hybrid_target if hybrid else _dense_target)(make, case, physical, len(table), len(shape), 0)
        gpu.buffer(verify.PAGE_TABLE).upload(table)
        rows = sum(r for r, _ in shape)
        self.tokens = np.array(sum((make.chain(r, V) for r, _ in shape), []), np.uint32)
        self.uniforms = None
        if hybrid:
            lane = lambda i, parity, path: verify.HybridLane(*shape[i], table_first=first[i], pending_path=path, parity=parity)
            before = [lane(i, 1, 0) for i in range(len(shape))]
            gpu.set_block(before, make.rng.integers(0, V, rows).astype(np.uint32))
            torch.cuda.synchronize()
            make.backend.run(gpu.encode(before, commit=False))      # the step before: its tape holds the rows this one folds
            self.lanes = [lane(i, 0, (1 << shape[i][0]) - 1) for i in range(len(shape))]
        else:
            policy = dict(temperature=case["temperature"], min_p=0.02, top_k=64, top_p=0.95) if case["temperature"] else {}
            self.lanes = [verify.Lane(r, c, table_first=f, **policy) for (r, c), f in zip(shape, first)]
            if policy:
                self.uniforms = make.rng.random((rows, 2), dtype=np.float32)
                self._draft_distribution(make, shape, V)
        self.out = dict(logits=_values(gpu.buffer(verify.LOGITS), torch.float32, rows, V), hidden=_values(gpu.buffer(verify.HIDDEN, 0), torch.bfloat16, rows, H))
        attention_layers = case["layers"] // 4 if hybrid else case["layers"]
        self.out["scales"] = _cached_scales(gpu, attention_layers, 2 * len(shape), m["kv_heads"], m["head_dim"])
        if hybrid:
            conv, kv = (2 * m["gdn_key_heads"] + m["gdn_value_heads"]) * 128, (m["gdn_key_heads"] + m["gdn_value_heads"]) * 128
            state = gpu.buffer(verify.GDN_STATES)
            self.out["state"] = [_strided(state, torch.float32, gpu.cell_offset(i, 1) + gpu.strides.convolution_state_bytes,
                                          (gpu.gdn_layers, m["gdn_value_heads"] * 128 * 128), (gpu.strides.recurrent_layer_bytes, 4))
                                 for i in range(len(shape))]
            self.out["carry"] = [_strided(state, torch.bfloat16, gpu.cell_offset(i, 1), (gpu.gdn_layers, 3 * conv), (gpu.strides.convolution_layer_bytes, 2))
                                 for i in range(len(shape))]
            self.out["tape"] = [_strided(gpu.buffer(verify.GDN_TAPE), torch.bfloat16, gpu.tape_offset(i, 0, 0), (gpu.gdn_layers, 16 * (conv + kv)),
                                         (gpu.tape_layer_bytes, 2)) for i in range(len(shape))]
        else:
            self.out["qkv"] = _values(gpu.buffer(verify.QKV_ROWS), torch.bfloat16, rows, (m["q_heads"] + 2 * m["kv_heads"]) * m["head_dim"])
            self.out["attention"] = _values(gpu.buffer(verify.ATTENTION_ROWS), torch.bfloat16, rows, m["q_heads"] * m["head_dim"])
        torch.cuda.synchronize()

    def _draft_distribution(self, make, shape, vocabulary):
        """What a draft model gives a sampled block: distributions with most of their mass on the drafted token."""
        drafted, at = np.zeros(len(self.tokens), np.int64), 0
        for rows, _ in shape:
            drafted[at:at + rows - 1] = self.tokens[at + 1:at + rows]
            drafted[at + rows - 1] = make.rng.integers(0, vocabulary)
            at += rows
        logits = torch.randn((len(drafted), vocabulary), device="cuda", generator=make.torch) * 1.5
        logits[torch.arange(len(drafted)), torch.from_numpy(drafted)] = 14.0
        _values(self.gpu.buffer(verify.DRAFT_PROBABILITIES), torch.float32, len(drafted), vocabulary).copy_(torch.softmax(logits, 1))

    def run(self):
        self.gpu.set_block(self.lanes, self.tokens, uniforms=self.uniforms)
        self.gpu.backend.run(self.gpu.encode(self.lanes, commit=True))
        tokens, retained, accepted, mask = self.gpu.results(self.lanes)
        kept, at = np.zeros_like(tokens), 0
        for i, lane in enumerate(self.lanes):      # only a lane's retained tokens are its results
            kept[at:at + retained[i]] = tokens[at:at + retained[i]]
            at += lane.rows
        return dict(self.out, tokens=kept, retained=retained, accepted=accepted, mask=mask)


class _Prefill:
    """A prompt chunk of one sequence through a target's layers."""

    def __init__(self, case, seed):
        make = _Maker(seed)
        hybrid = case["kind"] == "hybrid_prefill"
        m = HYBRID if hybrid else DENSE[case["model"]]
        tokens, self.committed = case["tokens"], case["committed"]
        count = -(-(self.committed + tokens) // PAGE)
        written = count - self.committed // PAGE
        table, physical, _ = _tables(make, [count], [written])
        self.gpu = gpu = (_hybrid_target if hybrid else _dense_target)(make, case, physical, len(table), 1, tokens)
        gpu.buffer(verify.PAGE_TABLE).upload(table)
        if not hybrid and case["staged"]:
            gpu.set_staged_prefill(True)
        self.tokens = np.array(make.chain(tokens, m["vocabulary"]), np.uint32)
        self.hybrid = hybrid
        self.out = dict(hidden=_values(gpu.buffer(verify.HIDDEN, 0), torch.bfloat16, tokens, m["hidden"]))
        attention_layers = case["layers"] // 4 if hybrid else case["layers"]
        self.out["scales"] = _cached_scales(gpu, attention_layers, written, m["kv_heads"], m["head_dim"])
        if hybrid:
            self.out["state"] = _strided(gpu.buffer(verify.GDN_STATES), torch.float32, gpu.cell_offset(0, 1) + gpu.strides.convolution_state_bytes,
                                         (gpu.gdn_layers, m["gdn_value_heads"] * 128 * 128), (gpu.strides.recurrent_layer_bytes, 4))
        torch.cuda.synchronize()

    def run(self):
        self.gpu.set_prefill_block(self.tokens)
        if self.hybrid:
            graph = self.gpu.encode_prefill(0, 0, self.committed, self.tokens.size)
        else:
            graph = self.gpu.encode_prefill(0, self.committed, self.tokens.size)
        self.gpu.backend.run(graph)
        return self.out


class _Draft:
    """The draft model's forward pass of its lanes' eight query rows."""

    def __init__(self, case, seed):
        make = _Maker(seed)
        H, F, L, V, lanes = DRAFT["hidden"], DRAFT["intermediate"], DRAFT["layers"], DRAFT["vocabulary"], case["lanes"]
        self.gpu = gpu = verify.DFlashDraft(make.backend, L, H, V, F, DRAFT["target_layers"], max_lanes=lanes)
        q4, rng = ops.FMT_Q4K, make.rng
        conv = lambda: make.bf16(np.stack([1 + 0.1 * rng.standard_normal(H), 0.2 * rng.standard_normal(H)] * 2))
        for layer in range(L):
            gpu.set_layer(layer, attention_dynamic=make.projection([(q4, H // 4)], H), qkv=make.projection([(q4, 6144)], H),
                          output=make.projection([(q4, H)], 4096, 0.005), mlp_dynamic=make.projection([(q4, H // 4)], H),
                          gate=make.projection([(q4, F)], H), up=make.projection([(q4, F)], H), down=make.projection([(q4, H)], F, _down_std(H, F)),
                          input_norm=make.norm(H), attention_convolution=conv(), query_norm=make.norm(128), key_norm=make.norm(128),
                          post_attention_norm=make.norm(H), mlp_convolution=conv())
        embedding, head = make.embedding_and_head(V, H)
        gpu.set_model(make.projection([(q4, H)], DRAFT["target_layers"] * H), make.norm(H), make.norm(H), make.projection([(q4, 256)], H),
                      make.norm(H), head)
        rings = gpu.buffer(verify.DFLASH_RINGS)
        make.normal(rings, torch.bfloat16, rings.size_bytes // 2, 0.5)
        self.cached = [max(0, case["cached"] - 101 * lane) for lane in range(lanes)]
        angle = (np.array(self.cached)[:, None, None] + np.arange(16)[None, :, None]) * 1e7 ** (-np.arange(64) / 64)
        gpu.buffer(verify.DFLASH_ROPE_COS).upload(np.cos(angle).astype(np.float32))
        gpu.buffer(verify.DFLASH_ROPE_SIN).upload(np.sin(angle).astype(np.float32))
        # a lane's first row is its anchor's embedding; the forward pass fills the others with the mask's
        hidden = gpu.buffer(verify.DFLASH_HIDDEN, 0)
        self.anchors = [(make.backend.from_array(rng.integers(0, V, 1).astype(np.uint32)), hidden.view(8 * lane * H * 2, H * 2)) for lane in range(lanes)]
        self.embedding, self.rows = embedding, 8 * lanes
        self.out = dict(logits=_values(gpu.buffer(verify.DFLASH_LOGITS), torch.float32, self.rows, V),
                        final=_values(gpu.buffer(verify.DFLASH_FINAL_HIDDEN), torch.bfloat16, self.rows, H),
                        selector=_values(gpu.buffer(verify.DFLASH_SELECTOR_HIDDEN), torch.bfloat16, self.rows, 256))
        torch.cuda.synchronize()

    def run(self):
        graph = splash_amd.CommandGraph()
        for anchor, row in self.anchors:
            ops.Embedding.add(graph, ops.FMT_Q4K, self.embedding, DRAFT["vocabulary"], DRAFT["hidden"], anchor, row, 1)
        self.gpu.backend.run(self.gpu.encode_decode(self.cached, graph=graph))
        return self.out


class _Select:
    """From a draft's logits to the rows a step verifies: candidates and edges, trees, the packed rows and their children."""

    def __init__(self, case, seed):
        make = _Maker(seed)
        self.backend, self.lanes, V = make.backend, case["lanes"], DRAFT["vocabulary"]
        L = self.lanes
        self.vocabulary, self.rows = V, 16 * L
        alloc = make.backend.allocate_buffer
        sizes = dict(logits=L * 8 * V * 4, hidden=L * 8 * 256 * 2, before=V * 256 * 2, after=V * 256 * 2, candidates=L * 7 * 16 * 4, unary=L * 7 * 16 * 4,
                     edges=L * 7 * 256 * 4, scratch=ops.DraftSelector.candidate_scratch_bytes(L, V), chain_tokens=L * 15 * 4, chain_rates=L * 15 * 16,
                     tokens=L * 64, trees=L * 128, scores=L * 128, sizes=max(16, L * 4), draws=L * 64, next=L * 1024, caps=L * 64, input=self.rows * 4,
                     tree_rows=self.rows * 8, lane_rows=max(16, L * 8), sources=self.rows * 4, ids=self.rows * 64, q=self.rows * 64, drawn=self.rows * 4,
                     depths=self.rows * 4)
        self.b = b = {name: alloc(size, label=name) for name, size in sizes.items()}
        make.normal(b["logits"], torch.float32, L * 8 * V, 2.0)
        make.normal(b["hidden"], torch.bfloat16, L * 8 * 256, 1.0)
        for book in ("before", "after"):
            make.normal(b[book], torch.bfloat16, V * 256, 0.08)
        self.tree_lanes = [dict(anchor=int(make.rng.integers(0, V)), depth=15, children=case["children"], intercept=[0.4] * 7,
                                temperature=0.7 if lane % 2 else 0.0, noise=int(make.rng.integers(0, 1 << 62))) for lane in range(L)]
        kinds = dict(candidates=torch.int32, unary=torch.float32, tokens=torch.int32, trees=torch.int32, scores=torch.float32, next=torch.float32,
                     input=torch.int32, tree_rows=torch.int32, ids=torch.int32, q=torch.float32, drawn=torch.uint8, depths=torch.int32)
        self.out = {name: _bytes(b[name]).view(kind) for name, kind in kinds.items()}
        edges = _bytes(b["edges"]).view(torch.float32).view(L, 7, 256)
        self.out["edges"] = [edges[:, 1:], edges[:, 0, :16]]      # the first position follows the anchor alone
        torch.cuda.synchronize()

    def run(self):
        b, g, V = self.b, splash_amd.CommandGraph(), self.vocabulary
        ops.DraftSelector.add_candidates(g, b["logits"], b["hidden"], b["scratch"], b["candidates"], b["unary"], b["edges"], b["before"], b["after"], V, V, V,
                                         [lane["anchor"] for lane in self.tree_lanes])
        ops.DraftSelector.add_tree(g, b["candidates"], b["unary"], b["edges"], b["chain_tokens"], b["chain_rates"], b["tokens"], b["trees"], b["scores"],
                                   b["sizes"], b["draws"], b["next"], b["caps"], self.tree_lanes)
        ops.DraftSelector.add_verify_row_slots(g, b["tokens"], b["trees"], b["scores"], b["sizes"], b["input"], b["tree_rows"], b["lane_rows"], b["sources"],
                                               self.lanes, 16)
        ops.DraftSelector.add_verify_children(g, b["sources"], b["lane_rows"], b["tree_rows"], b["candidates"], b["next"], b["draws"], b["ids"], b["q"],
                                              b["drawn"], b["depths"], self.lanes, self.rows)
        self.backend.run(g)
        return self.out


_KINDS = dict(dense=_Step, hybrid=_Step, prefill=_Prefill, hybrid_prefill=_Prefill, draft=_Draft, select=_Select)


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "select":
        V, L = DRAFT["vocabulary"], case["lanes"]
        # the proposal rows' logits once, the codebook rows of the candidates
        return dict(bytes=L * 7 * V * 4 + L * 7 * 17 * 2 * 512, flops=L * 7 * 256 * 256 * 3)
    if kind == "draft":
        H, F, V, rows = DRAFT["hidden"], DRAFT["intermediate"], DRAFT["vocabulary"], 8 * case["lanes"]
        weights = DRAFT["layers"] * (2 * H * H // 4 + 6144 * H + H * 4096 + 3 * F * H) + 256 * H
        window = sum(min(2048, max(0, case["cached"] - 101 * lane)) for lane in range(case["lanes"]))
        ring = DRAFT["layers"] * window * 2 * 1024 * 2
        return dict(bytes=weights * Q4 + V * H * Q6 + ring + rows * V * 4, flops=2 * rows * (weights + V * H) + DRAFT["layers"] * window * 8 * 4 * 4096)
    hybrid = kind.startswith("hybrid")
    m = HYBRID if hybrid else DENSE[case["model"]]
    H, V, D, QH, KVH, layers = m["hidden"], m["vocabulary"], m["head_dim"], m["q_heads"], m["kv_heads"], case["layers"]
    step = kind in ("dense", "hybrid")
    lanes = _lanes(case) if step else [(case["tokens"], case["committed"])]
    rows = sum(r for r, _ in lanes)
    token = KVH * (2 * D + 4)      # an INT8 token's keys and values and their scales
    attends = layers // 4 if hybrid else layers
    size = attends * sum(r + c for r, c in lanes) * token
    flops = attends * sum(4.0 * QH * D * r * (c + (r + 1) / 2) for r, c in lanes)
    mixer = H * (2 * QH + 2 * KVH) * D      # q|k|v and the output projection
    if hybrid:
        VH, conv = m["gdn_value_heads"], (2 * m["gdn_key_heads"] + m["gdn_value_heads"]) * 128
        gdn = layers - attends
        gdn_mixer = H * (conv + VH * 128 + 2 * VH + VH * 128)
        hit = m["experts"] * (1 - (1 - m["top_k"] / m["experts"]) ** rows)
        expert = 3 * H * m["expert_ffn"]
        size += (attends * mixer + gdn * gdn_mixer + layers * hit * expert) * Q4 + layers * m["experts"] * H * Q6
        # a lane's recurrent state read and written, and the rows' inputs and keys, values on its tape
        size += gdn * (len(lanes) * 2 * VH * 128 * 128 * 4 + (rows * 2 * (conv + VH * 128) * 2 if step else 0))
        flops += 2.0 * rows * (attends * mixer + gdn * gdn_mixer + layers * (m["top_k"] * expert + m["experts"] * H))
        flops += gdn * rows * VH * 128 * 128 * (14 if step else 8)
    else:
        F = m["ffn"]
        size += layers * ((mixer + 2 * H * F) * Q4 + H * F * Q6)
        flops += 2.0 * rows * layers * (mixer + 3 * H * F)
    size += rows * H * Q4 + rows * H * 2
    if step:
        size += V * H * Q6 + rows * V * 4 * (2 if case.get("temperature") else 1)
        flops += 2.0 * rows * V * H
    return dict(bytes=float(size), flops=float(flops))


def tolerance(case):
    if case["kind"] == "select":
        return dict(rel=1e-4, max=1e-2, differ=0.002)      # fp32 sums of 256 products; equal ids and trees
    # rows rounded to 16 bits several times a layer, over up to eight layers
    return dict(rel=0.02, max=0.9)
