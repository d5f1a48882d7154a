"""The deposit's ways of summing a chunk of particles (a box of cells in LDS
with one to 64 copies, a hash table of cells, straight to the mesh) against the PM
oracle, by the extent of the particles and their number about the chunk's 1024."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import oracle_pm as op  # noqa: E402

pytestmark = pytest.mark.gpu

BITS = 2 ** 30


# extent in cells along x, y, z: 3^3 cells (64 copies), 5^3 (32), 8^3 (8), 2, 1 copies,
# past the tile (hash), everywhere in 64^3 cells (the hash table overflows)
@pytest.mark.parametrize("extent", [(1, 1, 1), (3, 3, 3), (6, 6, 6), (1, 1, 60), (10, 10, 14), (14, 14, 14), (15, 15, 15),
                                    (64, 20, 3), (64, 64, 64)])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 6000])
@pytest.mark.parametrize("tagged", [False, True])
def test_deposit_by_extent(gpu_ctx, extent, n, tagged):
    N, box = 64, 80.0
    g = np.random.default_rng(n + sum(extent))
    h = BITS // N
    lo = np.array([N - 2, 5, N - extent[2] // 2]) % N            # boxes across the periodic border too
    posi = (((lo + g.uniform(0, extent, (n, 3))) * h).astype(np.int64) % BITS).astype(np.int32)
    tag = (g.uniform(size=n) < 0.6).astype(np.int32) if tagged else None
    print(f"case: extent={extent} n={n} tagged={tagged}", flush=True)
    rs = 1.25 * box / N
    gpu_ctx.pm_forces(posi, tag, box / BITS, box, N, rs, 0.37)
    _, rho, _ = op.pm_forces(posi, tag, box / BITS, np.float32(box), N, np.float32(rs), np.float32(0.37))
    # the same FP32 products summed in FP64 in another order: 6000 2^-53 of a cell's sum
    np.testing.assert_allclose(gpu_ctx.pm_mesh(0), rho, rtol=1e-12, atol=1e-12 * max(rho.max(), 1e-30))
