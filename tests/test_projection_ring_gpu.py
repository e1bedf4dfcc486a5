"""The decode projection's ring of staged rows at the ends of its ranges (kernels/gguf_linear.hip)."""
import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc
from tests.test_gguf_gpu import ALL_FORMATS, run_projection
from tests.test_gguf_gpu import test_gate_up_table_epilogue_equals_the_table_pass as gate_up_table
from tests.test_gguf_gpu import test_residual_norm_epilogue as residual_norm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ALL_FORMATS)
@pytest.mark.parametrize("blocks", [1, 2, 3, 5])
def test_short_ranges_at_every_height(backend, fmt, blocks):
    """A workgroup's range of one to five super-blocks (the ring is filled past its end, and ends on either of its records),
    whole and in parts of one super-block, at the edges of the row tiles and with a wave past the last column tile: within
    the oracle's bound of the 64-bit sums, and every row the bits it has in the tallest block."""
    rng = np.random.default_rng(blocks)
    N, K = 80, 256 * blocks
    native = orc.make_native(fmt, N, K, 9 + blocks)
    x = orc.f32_to_bf16(rng.standard_normal((64, K)).astype(np.float32))
    linear = ops.Linear(backend)
    want = orc.gemm(fmt, native, x, N)
    for splits in sorted({1, blocks}):
        print(f"case ring fmt={fmt} blocks={blocks} splits={splits}", flush=True)
        full, _, _ = run_projection(backend, linear, fmt, [(N, native)], K, x, float32=True, splits=splits, whole_groups=0)
        assert np.all(np.abs(full.astype(np.float64) - want["exact"]) <= want["bound"])
        for rows in (1, 16, 17, 32, 33, 48):
            part, _, _ = run_projection(backend, linear, fmt, [(N, native)], K, x[:rows], float32=True, splits=splits, whole_groups=0)
            assert part.tobytes() == full[:rows].tobytes(), rows


@pytest.mark.parametrize("M", [33, 40, 48])
def test_three_row_tiles_write_what_four_do(backend, M):
    """Steps of 33 to 48 rows: the residual and gate/up rows, whole and in parts, are those of a 64-row block bit for bit; the
    tables that gate/up and the norming residual leave are held to what they are at other heights."""
    print(f"case three row tiles M={M}", flush=True)
    rng = np.random.default_rng(M)
    N, K = 320, 1280
    linear = ops.Linear(backend)
    for fmt in (ops.FMT_Q4K, ops.FMT_Q6K):
        native, gate = orc.make_native(fmt, N, K, 70), orc.make_native(fmt, N, K, 71)
        x, residual = (orc.f32_to_bf16(rng.standard_normal((64, width)).astype(np.float32)) for width in (K, N))
        for splits, whole in ((1, 0), (3, 1)):
            for extra in (dict(epilogue=ops.EPILOGUE_RESIDUAL, residual_bits=residual), dict(epilogue=ops.EPILOGUE_GATE_UP, gate_native=gate)):
                full, _, _ = run_projection(backend, linear, fmt, [(N, native)], K, x, splits=splits, whole_groups=whole, **extra)
                if "residual_bits" in extra:
                    extra["residual_bits"] = residual[:M]
                part, _, _ = run_projection(backend, linear, fmt, [(N, native)], K, x[:M], splits=splits, whole_groups=whole, **extra)
                assert part.tobytes() == full[:M].tobytes()
    gate_up_table(backend, M)
    for fmt, n, k, config in ((ops.FMT_Q4K, 512, 768, None), (ops.FMT_Q6K, 512, 2048, None)):
        residual_norm(backend, fmt, n, k, M, config)


@pytest.mark.parametrize("fmt", [f for f in ALL_FORMATS if f not in (ops.FMT_Q4K, ops.FMT_Q6K)])
def test_three_row_tiles_of_the_other_formats(backend, fmt):
    """The same of the formats with other records: the residual and gate/up rows of 40 are a 64-row block's, the norming residual
    is held to its rows, and gate/up's table, rows and what they are projected to are those of a table pass of its own."""
    print(f"case three row tiles fmt={fmt}", flush=True)
    rng = np.random.default_rng(fmt)
    M, N, K = 40, 320, 1280
    linear = ops.Linear(backend)
    native, gate = orc.make_native(fmt, N, K, 70), orc.make_native(fmt, N, K, 71)
    x, residual = (orc.f32_to_bf16(rng.standard_normal((64, width)).astype(np.float32)) for width in (K, N))
    for splits, whole in ((1, 0), (3, 1)):
        config = dict(splits=splits, whole_groups=whole)
        for epilogue, extra in ((ops.EPILOGUE_RESIDUAL, lambda rows: dict(residual_bits=residual[:rows])), (ops.EPILOGUE_GATE_UP, lambda rows: dict(gate_native=gate))):
            part, full = (run_projection(backend, linear, fmt, [(N, native)], K, x[:rows], epilogue=epilogue, **config, **extra(rows))[0] for rows in (M, 64))
            assert part.tobytes() == full[:M].tobytes()
    residual_norm(backend, fmt, 512, 768, M, None)
    residual_norm(backend, fmt, 512, 1024, M, (4, 3))
    hidden, ffn = 512, 768
    pair = [ops.Projection.from_native(backend, [(fmt, ffn, orc.make_native(fmt, ffn, hidden, seed))], hidden) for seed in (5, 6)]
    down = ops.Projection.from_native(backend, [(fmt, hidden, orc.make_native(fmt, hidden, ffn, 7))], ffn)
    rows, res = (backend.from_array(orc.f32_to_bf16(rng.standard_normal((M, hidden)).astype(np.float32))) for _ in range(2))
    got = []
    for fused in (False, True):
        scratch = ops.LinearScratch(backend, *[max(linear.scratch_size(*s, M)[i] for s in ((ffn, hidden), (hidden, ffn))) for i in range(3)])
        table = backend.allocate_buffer(ops.gguf_table_bytes(ffn, M)) if fused else None
        mid, out, graph = backend.allocate_buffer(M * ffn * 2), backend.allocate_buffer(M * hidden * 2), splash_amd.CommandGraph()
        linear.add_swiglu(graph, *pair, down, rows, mid, res, out, M, scratch, next_table=table)
        assert f"m48_{'gt' if fused else 'g'}" in " ".join(graph.kernels())
        backend.run(graph)
        got.append([mid.download(np.uint16), out.download(np.uint16), (table if fused else scratch.table).download(np.uint8)[:ops.gguf_table_bytes(ffn, M)]])
    for apart, together in zip(*got):
        assert np.array_equal(apart, together)
