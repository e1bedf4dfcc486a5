"""The decode projection's ring of staged rows at the ends of its ranges (kernels/gguf_linear.hip)."""
import numpy as np
import pytest

from splash_amd import ops
from tests import oracle as orc
from tests.test_gguf_gpu import ALL_FORMATS, run_projection

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
