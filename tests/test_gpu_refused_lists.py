"""A refused list: pp2p_set_tasks has dropped the old list, so that the next
evaluation is that of an empty one; pp2p_add_tasks leaves the list as it was."""
import ctypes

import numpy as np
import pytest

import photons_p2p as pp
from test_zz_no_alloc import _hip_lib

pytestmark = pytest.mark.gpu


def _context(ctx):
    g = np.random.default_rng(3)
    ctx.set_tuning()
    ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    ctx.set_particles(g.random((70, 3)), (10 * np.arange(7)).astype(np.int32), np.full(7, 10, np.int32))
    t, s = g.integers(0, 7, 40).astype(np.int32), g.integers(0, 7, 40).astype(np.int32)
    ctx.set_tasks(t, s)
    ctx.compute()
    return t, s, ctx.acc()


@pytest.mark.parametrize("form", [pp.EXEC_QUEUE, pp.EXEC_GRID, pp.EXEC_PER_TARGET])
def test_refused_set_tasks_leaves_an_empty_list(gpu_ctx, form):
    t, s, want = _context(gpu_ctx)
    assert np.abs(want).max() > 0
    bad = t.copy()
    bad[17] = 7
    with pytest.raises(pp.P2PError, match="task 17 "):
        gpu_ctx.set_tasks(bad, s)
    gpu_ctx.zero_acc()
    gpu_ctx.compute(form)
    assert np.all(gpu_ctx.acc() == 0.0)
    stats = gpu_ctx.list_stats()
    assert stats["ntask"] == stats["nrows"] == stats["nitems"] == stats["npairs"] == 0
    gpu_ctx.set_tasks(t, s)
    gpu_ctx.compute(form)
    assert np.allclose(gpu_ctx.acc(), want, rtol=1e-12, atol=0)


def test_refused_add_tasks_leaves_the_list(gpu_ctx):
    t, s, want = _context(gpu_ctx)
    bad = s.copy()
    bad[3] = -1
    with pytest.raises(pp.P2PError, match="task 3 "):
        gpu_ctx.add_tasks(t, bad)
    gpu_ctx.zero_acc()
    gpu_ctx.compute()
    assert np.allclose(gpu_ctx.acc(), want, rtol=1e-12, atol=0)


@pytest.mark.parametrize("n", [300000, 8 << 20])
def test_a_refused_list_takes_no_memory(n):
    """The ids are checked before the arrays grow, also those of a list that has
    to be appended to another one."""
    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert _hip_lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    with pp.Context(0) as ctx:
        t, s, want = _context(ctx)
        bad = np.zeros(n, np.int32)
        bad[n - 1] = 7
        before = free()
        for put in (ctx.add_tasks, ctx.set_tasks):
            with pytest.raises(pp.P2PError, match=f"task {n - 1} "):
                put(np.zeros(n, np.int32), bad)
        assert free() > before - 8 * n // 2                  # two arrays of n would take 8 n bytes
        ctx.set_tasks(t, s)
        ctx.zero_acc()
        ctx.compute()
        assert np.allclose(ctx.acc(), want, rtol=1e-12, atol=0)
