"""The device time of the multipole pass: its three parts (upward, M2L, downward)
are timed by the same events one after the other."""
import numpy as np
import pytest

import photons_p2p as pp

pytestmark = pytest.mark.gpu


def test_device_time_adds_the_three_passes(gpu_ctx):
    g = np.random.default_rng(6)
    p = g.integers(0, 1 << 28, (60000, 3)).astype(np.int32)
    x = p.astype(np.float64) * 1e-7
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    b = (x.min(0) - 1e-3).astype(np.float32), (x.max(0) + 1e-3).astype(np.float32)
    nl, nn = gpu_ctx.build_tree(p, np.ones(60000, np.int32), 1e-7, 16, *b)
    none = np.zeros(0, np.int32)
    gpu_ctx.fmm_short(none, none)
    empty = min(gpu_ctx.fmm_short(none, none) for _ in range(5))
    t, s = g.integers(0, nl + nn, (2, 3000000)).astype(np.int32)
    full = min(gpu_ctx.fmm_short(t, s) for _ in range(3))
    assert 0.0 < empty < full
