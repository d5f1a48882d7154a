"""The device tree at the edges of its two forms (device-wide levels above 4096
particles, one workgroup per subtree below) against the host builder, array
for array; and the multipoles on such a tree, whose levels and subtrees the
upward pass visits in different kernels, against the reference's operators."""
import numpy as np
import pytest

import photons_p2p as pp
import pyoracle as po
from photons_p2p import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("perm", "leaf_ip", "leaf_np", "active", "leaf_center", "leaf_width", "node_son", "node_center", "node_width")


def _posi(kind, n, g):
    if kind == "uniform":
        return g.integers(-(1 << 24), 1 << 28, (n, 3))              # ghosts lie below zero
    if kind == "clumps":                                            # unbalanced splits: small leaves beside large segments
        c = g.integers(1 << 26, 1 << 28, (40, 3))
        return c[g.integers(0, 40, n)] + (g.standard_cauchy((n, 3)) * 3e4).clip(-1e7, 1e7).astype(np.int64)
    if kind == "lattice":                                           # planes of equal coordinates
        m = int(round(n ** (1 / 3))) + 1
        q = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
        return 1000003 * (q + 1)
    p = g.integers(0, 1 << 28, (n, 3))                              # "coincident": a third of them in one point
    p[: n // 3] = p[0]
    return p


def _same(ctx, posi, int2pos, maxleaf, seed):
    g = np.random.default_rng(seed)
    n = posi.shape[0]
    posi = np.ascontiguousarray(posi[g.permutation(n)], np.int32)
    tag = (g.random(n) < 0.7).astype(np.int32)
    x = posi.astype(np.float64) * int2pos
    bdl, bdr = (x.min(0) - 1e-3).astype(np.float32), (x.max(0) + 1e-3).astype(np.float32)
    host = W.build_lists(posi, tag, int2pos, maxleaf, np.float32(0.5), np.float32(1.0), bdl, bdr, walk=False, with_tree=True)
    ctx.set_tuning()
    ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    nl, nn = ctx.build_tree(posi, tag, int2pos, maxleaf, bdl, bdr)
    dev = ctx.get_tree()
    assert (nl, nn) == (host["leaf_ip"].size, host["node_son"].shape[0])
    for k in KEYS:
        np.testing.assert_array_equal(dev[k], host[k], err_msg=k)
    return posi, tag, host


# grid steps: 53 significant bits, few (halfway cases in the sums of the means), one (exact sums)
STEPS = (1.7e-7, 138.671875 / (1 << 30), 2.0 ** -22)


@pytest.mark.parametrize("kind,n,maxleaf", [
    ("uniform", 4095, 32), ("uniform", 4096, 1), ("uniform", 4097, 1), ("uniform", 8193, 64), ("uniform", 4096, 4096),
    ("uniform", 9000, 4095), ("uniform", 20000, 5000), ("uniform", 350001, 48), ("clumps", 5000, 1), ("clumps", 60000, 7),
    ("clumps", 250000, 64), ("lattice", 4000, 1), ("lattice", 4096, 8), ("lattice", 30000, 1), ("coincident", 200, 64),
    ("coincident", 1500, 600), ("coincident", 9000, 3000)])
def test_tree_sizes(gpu_ctx, kind, n, maxleaf):
    print(f"case: {kind} n={n} maxleaf={maxleaf}", flush=True)
    g = np.random.default_rng(n + maxleaf)
    posi = _posi(kind, n, g)
    for step in STEPS:
        _same(gpu_ctx, posi, step, maxleaf, n)


def test_too_deep_is_refused(gpu_ctx):
    """More coincident particles than the depth limit can peel off one by one:
    an error, as before, and the context works on."""
    g = np.random.default_rng(1)
    posi = np.full((1500, 3), 12345, np.int32)
    tag = np.ones(1500, np.int32)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    b = np.float32([0, 0, 0]), np.float32([1, 1, 1])
    with pytest.raises(pp.P2PError):
        gpu_ctx.build_tree(posi, tag, 1e-6, 16, *b)
    with pytest.raises(pp.P2PError):
        gpu_ctx.walk_tree(0.5, 1.0)
    _same(gpu_ctx, _posi("uniform", 5000, g), 1.7e-7, 32, 7)


@pytest.mark.parametrize("kind,n,maxleaf", [("clumps", 9000, 16), ("uniform", 3000, 24)])
def test_multipoles_of_levels_and_subtrees(gpu_ctx, kind, n, maxleaf):
    g = np.random.default_rng(n)
    print(f"case: multipoles {kind} n={n}", flush=True)
    int2pos, mass = 1.7e-7, 0.37
    posi, tag, T = _same(gpu_ctx, _posi(kind, n, g), int2pos, maxleaf, n)
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0, mass=mass))
    gpu_ctx.build_tree(posi, tag, int2pos, maxleaf, *[(f(posi.astype(np.float64) * int2pos, 0) + s).astype(np.float32)
                                                     for f, s in ((np.min, -1e-3), (np.max, 1e-3))])
    nl, nn = T["leaf_ip"].size, T["node_son"].shape[0]
    # one local expansion handed down from the root's son pairs
    mt = np.array([nl] * 3 + [nl + nn // 2] * 2, np.int32)
    ms = np.array([0, nl - 1, nl + nn - 1, 1, nl - 2], np.int32)
    gpu_ctx.fmm_short(mt, ms)
    M, L = gpu_ctx.get_expansions()
    p = posi[T["perm"]]
    center = np.concatenate([T["leaf_center"], T["node_center"]])
    son = T["node_son"]
    cell = lambda sn: nl + sn if sn >= 0 else -sn - 1  # noqa: E731
    ref = np.zeros((nl + nn, 20), np.float32)
    for l in range(nl):
        a, c = T["leaf_ip"][l], T["leaf_np"][l]
        ref[l] = po.p2m_ref32(p[a:a + c], int2pos, T["leaf_center"][l], mass)
    for k in range(nn - 1, -1, -1):
        acc = np.zeros(20, np.float32)
        for sn in son[k]:
            acc = po.m2m_ref32(center[nl + k] - center[cell(sn)], ref[cell(sn)], acc)
        ref[nl + k] = acc
    assert np.array_equal(M, ref)
    Lf = po.m2l_tasks_f64(center.astype(np.float64), M.astype(np.float64), mt, ms, 1.0)
    for k in range(nn):
        for sn in son[k]:
            Lf[cell(sn)] = po.l2l_f64(center[cell(sn)].astype(np.float64) - center[nl + k].astype(np.float64),
                                      Lf[nl + k], Lf[cell(sn)])
    scale = np.abs(Lf).max(0) + 1e-30
    assert np.all(np.abs(L - Lf) <= 5e-5 * scale)


# means over several tiles: about the sampled strides (1, then 2) and a whole tile,
# with coordinates of both signs (sums that cross zero) or far from it
@pytest.mark.parametrize("n", [8191, 8192, 12289, 199999, 200000, 200001])
@pytest.mark.parametrize("offset", [0, 1 << 29])
def test_means_over_tiles(gpu_ctx, n, offset):
    print(f"case: n={n} offset={offset}", flush=True)
    g = np.random.default_rng(n)
    posi = g.integers(-(1 << 27), 1 << 27, (n, 3)) + offset
    for k, step in enumerate(STEPS):
        _same(gpu_ctx, posi, step, 1000, n + k)


# one subtree whose segments end at, before and after a batch of the threads' chains
# (8), a wave's 64 values and the longest chain of a wave (1024)
@pytest.mark.parametrize("n", [3, 15, 16, 17, 63, 64, 65, 127, 200, 1023, 1024, 1025, 2051])
@pytest.mark.parametrize("offset", [0, 1 << 29])
def test_segment_chains(gpu_ctx, n, offset):
    print(f"case: n={n} offset={offset}", flush=True)
    g = np.random.default_rng(n)
    posi = g.integers(-(1 << 27), 1 << 27, (n, 3)) + offset
    for k, step in enumerate(STEPS):
        _same(gpu_ctx, posi, step, 1, n + k)
