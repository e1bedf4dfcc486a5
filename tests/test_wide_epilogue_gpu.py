"""The wide projections' stores of two columns at once, wherever a destination begins (kernels/gguf_wide.hip)."""
import numpy as np
import pytest

import splash_amd
from splash_amd import ops
from tests import oracle as orc
from tests.test_wide_kernels_gpu import FORMATS, add_table, project, rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("rows", [1, 61, 64])
def test_rows_of_an_odd_place_and_stride(backend, name, rows):
    """Destination and residual one element into their buffers, rows an odd number of elements apart, the last tile's rows
    odd and even in number: the values of aligned rows, and nothing written beside them."""
    fmt, K, N, T = FORMATS[name], 512, 144, 4
    print(f"case wide epilogue {name} rows={rows}", flush=True)
    rng = np.random.default_rng(rows)
    stride = N + 1
    image = backend.from_array(ops.pack_gguf_image(fmt, orc.make_native(fmt, N, K, rows), N, K))
    residual = orc.f32_to_bf16(rng.standard_normal((rows, N)).astype(np.float32))
    graph = splash_amd.CommandGraph()
    table = add_table(graph, backend, rows_of(rng, rows, K))
    backend.run(graph)
    spread = np.zeros(rows * stride + 2, dtype=np.uint16)
    spread[1:-1].reshape(rows, stride)[:, :N] = residual
    for kind in ("a", "r"):
        near, far = backend.allocate_buffer(rows * N * 2), backend.allocate_buffer(spread.nbytes)
        far.fill(0x5A)
        project(backend, f"{name}_t{T}_{kind}", [image], [N], table, near, rows, K, T, residual=backend.from_array(residual))
        project(backend, f"{name}_t{T}_{kind}", [image], [N], table, far.view(2, spread.nbytes - 2), rows, K, T,
                residual=backend.from_array(spread).view(2, spread.nbytes - 2), stride=stride)
        got = far.download(np.uint16)
        assert got[0] == 0x5A5A and got[-1] == 0x5A5A
        got = got[1:-1].reshape(rows, stride)
        assert np.array_equal(got[:, :N], near.download(np.uint16).reshape(rows, N)) and np.all(got[:, N:] == 0x5A5A)
