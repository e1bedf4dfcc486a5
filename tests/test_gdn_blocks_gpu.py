"""The GDN prompt scan in blocks of sixteen tokens (gdn_prefill_blocks, gdn_prefill_block_scan) against 64-bit arithmetic
and against the token-by-token scan."""
import numpy as np
import pytest

import splash_amd
from tests import oracle as orc
from tests.gdn_case import check_prefill_against_fp64, make_rows, make_state
from tests.test_gdn_gpu import Chunk, Layer

pytestmark = pytest.mark.gpu


class BlockChunk(Chunk):
    """The chunk through the blocks; everything else as Chunk does it."""

    def run(self, packed, lane, current, nxt, captures=(), tiled_heads=False):
        gdn = self.layer.gdn
        blocks = self.layer.backend.allocate_buffer(gdn.prefill_blocks_bytes(packed.shape[0]))
        plain = type(gdn).add_prefill
        gdn.add_prefill = lambda *a, **k: plain(gdn, *a, blocks=blocks, **k)
        try:
            return super().run(packed, lane, current, nxt, captures, tiled_heads)
        finally:
            del gdn.add_prefill


def _recurrence(shape, got, state):
    """The recurrence in fp64 over the passes' own rows: outputs and the state after."""
    f = lambda bits: orc.bf16_to_f32(np.asarray(bits)).astype(np.float64)
    kh, vh, per = shape.key_heads, shape.value_heads, shape.value_heads // shape.key_heads
    q, k, v, beta = f(got["queries"]), f(got["keys"]), f(got["values"]), f(got["beta"])
    S, rows = state.astype(np.float64).copy(), np.zeros((q.shape[0], vh, 128))
    for t in range(q.shape[0]):
        kt, qt = (np.repeat(x[t].reshape(kh, 128), per, axis=0) for x in (k, q))
        S *= got["decay"][t].astype(np.float64)[:, None, None]
        delta = (v[t].reshape(vh, 128) - np.einsum("hrc,hc->hr", S, kt)) * beta[t][:, None]
        S += delta[:, :, None] * kt[:, None, :]
        rows[t] = np.einsum("hrc,hc->hr", S, qt)
    return rows, S


def _case(backend, heads, tokens, seed, shape_rows=None):
    rng = np.random.default_rng(seed)
    layer = Layer(backend, rng, *heads, lanes=1, cells=5)
    conv_in, state_in = make_state(rng, layer.shape)
    packed = make_rows(rng, layer.shape, tokens)
    if shape_rows:
        packed = shape_rows(layer.shape, packed)
    layer.write_cell(0, 0, conv_in, state_in)
    return layer, packed, conv_in, state_in


@pytest.mark.parametrize("heads,tokens", [((2, 4), 1), ((2, 4), 15), ((2, 2), 16), ((2, 4), 17), ((1, 3), 33), ((16, 32), 64), ((4, 8), 131), ((2, 2), 2048)])
def test_blocks_pass_the_scans_checks_and_lose_no_precision(backend, heads, tokens):
    print(f"case gdn blocks heads={heads} tokens={tokens}", flush=True)
    layer, packed, conv_in, state_in = _case(backend, heads, tokens, 51)
    scan = Chunk(layer, tokens).run(packed, 0, 0, 1)
    got = BlockChunk(layer, tokens).run(packed, 0, 0, 1)
    check_prefill_against_fp64(layer.shape, layer.conv_w, layer.a_scale, layer.dt_bias, layer.norm, packed, conv_in, state_in, got)
    for name in ("queries", "keys", "values", "decay", "beta", "conv_out"):
        assert got[name].tobytes() == scan[name].tobytes(), name
    rows, state = _recurrence(layer.shape, scan, state_in)
    off = lambda run: np.linalg.norm(run["state_out"] - state) / np.linalg.norm(state)
    error = lambda run: np.linalg.norm(orc.bf16_to_f32(run["recurrent"]).reshape(rows.shape) - rows) / np.linalg.norm(rows)
    print(f"  state off by {off(got):.3g} (scan {off(scan):.3g}), rows by {error(got):.5g} (scan {error(scan):.5g})", flush=True)
    # measured, state: 16 / 32 heads 4.97e-8 (scan 5.74e-8), of 2 to 4 heads 2.97e-8 .. 5.84e-8 (4.01e-8 .. 6.02e-8); two heads of
    # few rounded gates scatter by a tenth around that, which half a step of fp32 allows for
    assert off(got) <= max(1.05 * off(scan), 2.0 ** -24) and error(got) <= 1.001 * error(scan)


def test_blocks_of_equal_keys_and_of_vanishing_decays(backend):
    """The triangular system at its worst (every key of a block the same, betas near 1, no decay) and decays that underflow."""
    def gates(shape):
        at = shape.conv_dim + shape.value_heads * 128
        return slice(at, at + shape.value_heads), slice(at + shape.value_heads, at + 2 * shape.value_heads)

    def alike(shape, packed):
        f = orc.bf16_to_f32(packed)
        f[:, :shape.conv_dim - shape.value_heads * 128] = f[:1, :shape.conv_dim - shape.value_heads * 128]
        b, a = gates(shape)
        f[:, b] = 6.0       # beta near 1
        f[:, a] = -20.0     # softplus near 0: decay near 1
        return orc.f32_to_bf16(f)

    def vanishing(shape, packed):
        f = orc.bf16_to_f32(packed)
        f[3::7, gates(shape)[1]] = 400.0     # decay exp(-|a| 400) = 0
        return orc.f32_to_bf16(f)

    for name, change in (("alike", alike), ("vanishing", vanishing)):
        print(f"case gdn blocks {name}", flush=True)
        layer, packed, conv_in, state_in = _case(backend, (2, 4), 45, 52, change)
        scan = Chunk(layer, 45).run(packed, 0, 0, 1)
        got = BlockChunk(layer, 45).run(packed, 0, 0, 1)
        rows, state = _recurrence(layer.shape, scan, state_in)
        off = lambda run: np.linalg.norm(run["state_out"] - state) / np.linalg.norm(state)
        print(f"  state off by {off(got):.3g} (scan {off(scan):.3g})", flush=True)
        # a correction passes at most fifteen fp32 steps of a system whose entries are at most 1
        assert off(got) <= max(2 * off(scan), 16 * 2.0 ** -24)


def test_blocks_in_runs_and_refusals(backend):
    """Runs between captures continue one another, each run's blocks starting at its first row."""
    layer, packed, _, state_in = _case(backend, (2, 4), 45, 53)
    whole = BlockChunk(layer, 45).run(packed, 0, 0, 1)
    runs = BlockChunk(layer, 45).run(packed, 0, 0, 1, captures=[(7, 2), (32, 3)])
    scale = np.abs(whole["state_out"]).max()
    assert np.abs(runs["state_out"] - whole["state_out"]).max() <= 2e-6 * scale
    # the outputs of every run: bf16 of sums as far apart as the states, each row the gate pass's of its own values, and the
    # runs' own convolution carry
    wide = lambda run: orc.bf16_to_f32(run["recurrent"])
    assert np.all(np.abs(wide(runs) - wide(whole)) <= 0.0078125 * np.abs(wide(whole)) + 1e-5)
    same = (runs["recurrent"] == whole["recurrent"]).reshape(45, 4, 128).all(axis=2)
    assert same[7:32].mean() > 0.9 and same[32:].mean() > 0.9
    assert np.array_equal(runs["hidden"].reshape(45, 4, 128)[same], whole["hidden"].reshape(45, 4, 128)[same])
    assert runs["conv_out"].tobytes() == whole["conv_out"].tobytes()
    _, state = layer.read_cell(0, 3)
    alone = Chunk(layer, 32).run(packed[:32], 0, 0, 1)
    assert np.abs(state - alone["state_out"]).max() <= 2e-6 * scale
    graph = splash_amd.CommandGraph()
    buffers = dict(packed=backend.from_array(packed), states=layer.states, **layer.weights, **layer.gdn.prefill_workspace(backend, 45))
    small = backend.allocate_buffer(layer.gdn.prefill_blocks_bytes(45) - 16)
    with pytest.raises(ValueError):
        layer.gdn.add_prefill(graph, buffers, 0, 45, layer.cell(0, 0), layer.cell(0, 1), blocks=small)
    assert len(graph) == 0


@pytest.mark.parametrize("place", ["value", "key", "query", "beta", "decay", "infinite value", "infinite state", "state", "last row"])
def test_blocks_keep_what_is_not_finite_where_the_scan_keeps_it(backend, place):
    """Rows and states that are not finite reach through the blocks what they reach token by token, and nothing else: not the
    rows of their block before them, not the state's other rows. Where they reach, the sixteen state rows of a workgroup are
    the scan's bit for bit."""
    print(f"case gdn blocks not finite: {place}", flush=True)
    tokens, row, dimension = 45, 21, 37
    nan, inf = 0x7FC0, 0x7F80

    def change(shape, packed):
        packed, values = packed.copy(), 2 * shape.key_heads * 128
        gate = shape.conv_dim + shape.value_heads * 128
        at = {"value": values + 128 + dimension, "infinite value": values + 128 + dimension, "last row": values + 128 + dimension,
              "query": dimension, "key": (shape.key_heads + 1) * 128 + dimension, "beta": gate + 1, "decay": gate + shape.value_heads + 1}
        if place in at:
            packed[tokens - 1 if place == "last row" else row, at[place]] = inf if place == "infinite value" else nan
        return packed

    layer, packed, conv_in, state_in = _case(backend, (2, 4), tokens, 54, change)
    if "state" in place:
        state_in = state_in.copy()
        state_in[1, dimension, 5] = np.inf if place == "infinite state" else np.nan
        layer.write_cell(0, 0, conv_in, state_in)
    scan = Chunk(layer, tokens).run(packed, 0, 0, 1)
    got = BlockChunk(layer, tokens).run(packed, 0, 0, 1)
    widen = lambda run: (orc.bf16_to_f32(run["recurrent"]).reshape(tokens, 4, 128), run["state_out"])
    (rows, state), (want, want_state) = widen(got), widen(scan)
    broken = ~np.isfinite(want_state).all(axis=2)                   # [head][dimension]
    first = 0 if "state" in place else tokens - 1 if place == "last row" else row
    assert np.isfinite(want[:first]).all() and not np.isfinite(want[first:]).all()
    assert broken.any() == (place != "query") and not broken.all()
    for a, b in ((rows, want), (state, want_state)):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.where(np.isinf(a), a, 0), np.where(np.isinf(b), b, 0))
    groups = broken.reshape(4, 8, 16).any(axis=2)
    for head, group in zip(*np.nonzero(groups)):
        part = slice(16 * group, 16 * group + 16)
        assert rows[:, head, part].tobytes() == want[:, head, part].tobytes()
        assert state[head, part].tobytes() == want_state[head, part].tobytes()
    # elsewhere each form is within a bf16 step and 1e-5 of the recurrence (check_prefill_against_fp64's bound), its state within 1e-5
    finite, stays = np.isfinite(want), np.isfinite(want_state)
    assert np.all(np.abs(rows - want)[finite] <= 2 * (0.0078125 * np.abs(want[finite]) + 1e-5))
    assert np.abs(state - want_state)[stays].max() <= 2e-5
