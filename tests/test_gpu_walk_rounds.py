"""The rounds of the device walk where they can go wrong: more frames than the
arrays' first size (every leaf pair within the cutoff), a tree of one leaf, no
target at all, rounds at the edges of a tile, and the order of the
well-separated pairs (round by round, in frame order)."""
import numpy as np
import pytest

import photons_p2p as pp
from photons_p2p import workloads as W

pytestmark = pytest.mark.gpu


def _tree(n, maxleaf, theta, cutoff, seed, local=0.7):
    g = np.random.default_rng(seed)
    posi = g.integers(0, 1 << 28, (n, 3)).astype(np.int32)
    posi[: n // 3] = (posi[0] + g.normal(0, 4e6, (n // 3, 3))).clip(0, 1 << 29).astype(np.int32)
    tag = (g.random(n) < local).astype(np.int32)
    step = 1e-7
    x = posi.astype(np.float64) * step
    b = (x.min(0) - 1e-3).astype(np.float32), (x.max(0) + 1e-3).astype(np.float32)
    T = W.build_lists(posi, tag, step, maxleaf, np.float32(theta), np.float32(cutoff), *b, with_tree=True, with_m2l=True)
    return posi, tag, step, b, T


def _rounds(T, theta, cutoff):
    """Well-separated pairs of a level-by-level walk, as cells; FP32 as the reference."""
    f = np.float32
    nl = T["leaf_ip"].size
    C = lambda i: T["node_center"][i] if i >= 0 else T["leaf_center"][-i - 1]  # noqa: E731
    S = lambda i: T["node_width"][i] if i >= 0 else T["leaf_width"][-i - 1]  # noqa: E731
    cell = lambda i: nl + i if i >= 0 else -i - 1  # noqa: E731
    out, now = [], [(0, 0)]
    while now:
        nxt = []
        for i, j in now:
            if i < 0 and j < 0:
                continue
            if i == j:
                a, b = T["node_son"][i]
                nxt += [(a, a), (a, b), (b, a), (b, b)]
                continue
            w = (0.5 * (S(i) + S(j)).astype(np.float64)).astype(f)
            d = C(i) - C(j)
            m = np.maximum(np.abs(d) - w, f(0))
            acc = 0
            if float(f(f(m[0] + m[1]) + m[2])) >= 1e-15:
                if f(f(m[0] * m[0] + m[1] * m[1]) + m[2] * m[2]) > f(cutoff) * f(cutoff):
                    acc = -1
                else:
                    wm = f(2) * w.max()
                    dd = f(f(d[0] * d[0] + d[1] * d[1]) + d[2] * d[2])
                    acc = int(f(wm * wm) < f(f(f(theta) * f(theta)) * dd))
            if acc == 1:
                out.append((cell(i), cell(j)))
            elif acc == 0:
                si, sj = S(i), S(j)
                if i >= 0 and (j < 0 or f(f(si[0] + si[1]) + si[2]) > f(f(sj[0] + sj[1]) + sj[2])):
                    nxt += [(s, j) for s in T["node_son"][i]]
                else:
                    nxt += [(i, s) for s in T["node_son"][j]]
        now = nxt
    return out


@pytest.mark.parametrize("n,maxleaf,theta,cutoff", [
    (12000, 6, 0.01, 100.0),      # every leaf pair: several times the frames the arrays start with
    (3000, 16, 0.9, 4.0), (2000, 8, 0.6, 9.0), (5000, 40, 0.5, 3.0), (700, 700, 0.5, 1.0)])
def test_rounds_equal_the_host_walk(gpu_ctx, n, maxleaf, theta, cutoff):
    posi, tag, step, b, T = _tree(n, maxleaf, theta, cutoff, seed=n)
    print(f"case: n={n} maxleaf={maxleaf} theta={theta} tasks={T['task_t'].size} m2l={T['m2l_t'].size}", flush=True)
    with pp.Context(0) as ctx:                       # arrays of the first size
        ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
        ctx.build_tree(posi, tag, step, maxleaf, *b)
        for _ in range(2):                           # the second walk finds the arrays grown
            assert ctx.walk_tree(theta, cutoff) == T["task_t"].size
            tt, ts = ctx.get_tasks()
            np.testing.assert_array_equal(tt, T["task_t"])
            np.testing.assert_array_equal(ts, T["task_s"])
            mt, ms = ctx.get_m2l_tasks()
            assert mt.size == T["m2l_t"].size
            if n < 6000:
                assert list(zip(mt.tolist(), ms.tolist())) == _rounds(T, theta, cutoff)


@pytest.mark.parametrize("active", [0, -1])
def test_one_leaf(gpu_ctx, active):
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(np.random.default_rng(3).random((9, 3)), np.array([0], np.int32), np.array([9], np.int32))
    z = np.zeros((0, 3), np.float32)
    tree = {"node_son": np.zeros((0, 2), np.int32), "node_center": z, "node_width": z,
            "leaf_center": np.full((1, 3), 0.5, np.float32), "leaf_width": np.ones((1, 3), np.float32)}
    n = gpu_ctx.walk_tasks(tree, np.array([active], np.int32), 0.5, 1.0)
    assert n == (1 if active >= 0 else 0)
    tt, ts = gpu_ctx.get_tasks()
    assert tt.tolist() == ts.tolist() == [0] * n
    assert gpu_ctx.get_m2l_tasks()[0].size == 0


def test_no_targets(gpu_ctx):
    posi, tag, step, b, T = _tree(4000, 16, 0.5, 3.0, seed=8, local=0.0)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.build_tree(posi, tag, step, 16, *b)
    assert gpu_ctx.walk_tree(0.5, 3.0) == T["task_t"].size == 0
    assert gpu_ctx.get_m2l_tasks()[0].size == T["m2l_t"].size
