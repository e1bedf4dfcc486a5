"""The row passes at every workgroup size that is right for them: the operators' own, and the 256 threads a launch by name has
where it states none. Bit for bit the separate passes."""
import ctypes

import numpy as np
import pytest

import splash_amd
from splash_amd import _native as nat
from splash_amd import ops
from tests import oracle as orc
from tests.test_oracle_draft_tree import drawn_lattice

pytestmark = pytest.mark.gpu
U32 = ctypes.c_uint32


class Norm(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("width", "rows", "tiles", "reserved")]


class Prepare(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("input_size", "rows", "tiles", "row_stride")]


class Conv(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("finish", "hidden")]


class ConvTable(ctypes.Structure):
    _fields_ = [(n, U32) for n in ("hidden", "rows", "tiles")]


class Tree(ctypes.Structure):
    _fields_ = [(n, U32 * 8) for n in ("anchor", "depth", "chain", "children")] + [("lanes", U32), ("reserved", U32 * 3), (
        "slope", ctypes.c_float * 8), ("intercept", ctypes.c_float * 56), ("temperature", ctypes.c_float * 8), ("noise", U32 * 16)]


def row_threads(width):
    """norm_row_threads: a thread a vector of eight columns."""
    return 256 if width > 8192 or width <= 2048 else -(-width // 512) * 64


def bf16(backend, values):
    return backend.from_array(orc.f32_to_bf16(np.asarray(values, np.float32)))


def filled(backend, *sizes):
    return [backend.from_array(np.full(n, 0xA5, np.uint8)) for n in sizes]


# the narrowest row; one with a half-filled wave of vectors; past 256 vectors by half a wave; a draft's; the widest in LDS; past it
@pytest.mark.parametrize("width", [256, 768, 2304, 5120, 8192, 8448])
@pytest.mark.parametrize("rows", [1, 17])
def test_a_norm_with_its_table_at_every_workgroup_size(backend, rows, width):
    print(f"case norm threads rows={rows} width={width}", flush=True)
    rng = np.random.default_rng(width + rows)
    x, weight = bf16(backend, rng.standard_normal((rows, width))), bf16(backend, 1 + 0.2 * rng.standard_normal(width))
    tiles = (rows + 15) // 16
    sizes = rows * width * 2, ops.gguf_table_bytes(width, rows)
    want = filled(backend, *sizes)
    graph = splash_amd.CommandGraph()
    ops.Normalization.add_rms(graph, x, weight, want[0], width, rows)
    graph.add("gguf_prepare_table", [want[0], want[1]], Prepare(width, rows, tiles, width), (width // 32, tiles, 1), (64, 1, 1))
    got = {threads: filled(backend, *sizes) for threads in sorted({256, row_threads(width)} | ({512, 1024} if width <= 8192 else set()))}
    for threads, out in got.items():
        graph.add("norm_rms_table16", [x, weight, *out], Norm(width, rows, tiles, 0), (16 * tiles, 1, 1), (threads, 1, 1))
    backend.run(graph)
    for threads, out in got.items():
        for a, b in zip(want, out):
            assert np.array_equal(a.download(), b.download()), threads


@pytest.mark.parametrize("width", [256, 768, 2304, 5120, 8192])
@pytest.mark.parametrize("lanes", [1, 3])
def test_a_convolution_with_its_table_at_every_workgroup_size(backend, lanes, width):
    """Both stages: a workgroup of its own threads, and of 256 over the whole row; the rows of a tile past the live ones."""
    print(f"case convolution threads lanes={lanes} width={width}", flush=True)
    rng = np.random.default_rng(width + lanes)
    rows, groups = 8 * lanes, width // 16
    tiles = (rows + 15) // 16
    x, residual = (bf16(backend, rng.standard_normal((rows, width))) for _ in range(2))
    dynamic, base = bf16(backend, 0.3 * rng.standard_normal((rows, 4 * groups))), bf16(backend, rng.standard_normal((4, width)))
    weight = bf16(backend, 1 + 0.2 * rng.standard_normal(width))
    row_bytes, table_bytes = rows * width * 2, ops.gguf_table_bytes(width, rows)
    for finish in (0, 1):
        want = filled(backend, row_bytes, row_bytes, table_bytes)
        graph = splash_amd.CommandGraph()
        graph.add("draft_conv", [x, dynamic, base, residual if finish else x, want[0]], Conv(finish, width), (-(-8 * width // 256), lanes, 1))
        if finish:
            graph.add("norm_rms_table16", [want[0], weight, want[1], want[2]], Norm(width, rows, tiles, 0), (16 * tiles, 1, 1), (row_threads(width), 1, 1))
        else:
            graph.add("gguf_prepare_table", [want[0], want[2]], Prepare(width, rows, tiles, width), (width // 32, tiles, 1), (64, 1, 1))
        if finish:
            launches = [(1, threads) for threads in sorted({256, row_threads(width), 1024})]
        else:
            launches = [(-(-width // 512), 64), (1, 256), (2, 128)]
        got = []
        for across, threads in launches:
            out = filled(backend, row_bytes, row_bytes, table_bytes)
            graph.add("draft_conv_norm_table" if finish else "draft_conv_table", [x, dynamic, base, residual if finish else x, weight if finish else base,
                                                                               out[0], out[1] if finish else out[0], out[2]],
                      ConvTable(width, rows, tiles), (16 * tiles, across, 1), (threads, 1, 1))
            got.append(out)
        backend.run(graph)
        for launch, out in zip(launches, got):
            for a, b in zip(want, out):
                assert np.array_equal(a.download(), b.download()), (finish, launch)


@pytest.mark.parametrize("temperature", [0.0, 0.7])
def test_a_tree_is_the_same_by_fewer_threads(backend, temperature):
    print(f"case tree threads temperature={temperature}", flush=True)
    rng = np.random.default_rng(5)
    lanes = 8
    lattices = [drawn_lattice(rng) for _ in range(lanes)]
    inputs = [backend.from_array(np.concatenate([l[i] for l in lattices]).astype(dtype)) for i, dtype in enumerate((np.uint32, np.float32, np.float32))]
    chains = backend.from_array(rng.integers(0, 5000, (lanes, 15)).astype(np.uint32))
    rates = backend.from_array(rng.uniform(0, 0.9, (lanes, 15, 4)).astype(np.float32))
    params = Tree(lanes=lanes)
    for l in range(lanes):
        params.anchor[l], params.depth[l], params.chain[l], params.children[l] = l, 15 - l, 2 * l if l < 7 else 0, 1 + l % 4
        params.slope[l], params.temperature[l], params.noise[2 * l], params.noise[2 * l + 1] = 1.0 + 0.05 * l, temperature, 77 + l, l
    results = []
    for threads in (1024, 512, 256):
        out = filled(backend, lanes * 64, lanes * 128, lanes * 128, lanes * 4, lanes * 64, lanes * 16 * 64, lanes * 64)
        buffers = [*inputs, chains, rates, *out]
        handles = (ctypes.c_void_p * len(buffers))(*[b.handle for b in buffers])
        dispatch = nat.Dispatch(kernel=b"draft_select_tree", buffers=handles, buffer_count=len(buffers), params=ctypes.addressof(params),
                                params_bytes=ctypes.sizeof(params), grid=(U32 * 3)(lanes, 1, 1), block=(U32 * 3)(threads, 1, 1))
        ticket = ctypes.c_void_p()
        nat.check(nat.lib.sp_submit(backend.handle, ctypes.byref(dispatch), 1, None, None, ctypes.byref(ticket)))
        splash_amd.backend.Ticket(ticket.value).wait()
        results.append([b.download() for b in out])
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert np.array_equal(a, b)
