"""The largest list of pp2p_compute_noalloc: 32 bytes of its 64 MiB a task at
the sort (keys, sources, row marks and numbers, row targets and offsets, and two
copies of the sort's), 2.09 M tasks in all.  Just below it gives what pp2p_compute
gives, just above it is refused."""
import numpy as np
import pytest

import photons_p2p as pp
from test_zz_no_alloc import DevArray

pytestmark = pytest.mark.gpu

LIMIT = (64 << 20) // 32                     # 2097152 less what the queue head, alignment and the sort's counts take


@pytest.mark.parametrize("rows", [1, 1000])
@pytest.mark.parametrize("n,taken", [(LIMIT - 8192, True), (LIMIT + 1, False)])
def test_largest_list(gpu_ctx, n, taken, rows):
    print(f"case: compute_noalloc {n} tasks {rows} rows", flush=True)
    g = np.random.default_rng(n)
    nleaf = 1000
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(g.random((nleaf, 3)) * 5.0, np.arange(nleaf, dtype=np.int32), np.ones(nleaf, np.int32))
    t, s = (np.arange(n) % rows).astype(np.int32), g.integers(0, nleaf, n).astype(np.int32)
    dt, ds, acc = DevArray(t), DevArray(s), DevArray(np.zeros((3, nleaf)))
    try:
        if not taken:
            with pytest.raises(pp.P2PError, match="scratch"):
                gpu_ctx.compute_noalloc(n, dt.addr, ds.addr, acc.addr)
            return
        gpu_ctx.compute_noalloc(n, dt.addr, ds.addr, acc.addr)
        gpu_ctx.sync()
        got = acc.get().T
    finally:
        for d in (dt, ds, acc):
            d.free()
    gpu_ctx.set_tasks(t, s)
    gpu_ctx.compute()
    want = gpu_ctx.acc()
    # the order of the FP64 adds differs: a few thousand sums of partial sums
    assert np.abs(want).max() > 0 and np.abs(got - want).max() <= 1e-11 * np.abs(want).max()
