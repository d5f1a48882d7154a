"""Trees above one workgroup's 4096 particles in which one subtree of many does
not fit its workgroup (leaves of one particle and an empty leaf: more leaves than
particles), found after the level passes have moved the particles: the whole
tree is built again, level by level, and equals the host builder's array for array."""
import numpy as np
import pytest

import photons_p2p as pp
from photons_p2p import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("perm", "leaf_ip", "leaf_np", "active", "leaf_center", "leaf_width", "node_son", "node_center", "node_width")
STEP = 1.7e-7


def _misfits(T):
    """Largest subtrees of at most 4096 particles, and those with more leaves or nodes than particles."""
    son, nn = T["node_son"], T["node_son"].shape[0]
    part, leaves, nodes = (np.zeros(nn, np.int64) for _ in range(3))
    for k in range(nn - 1, -1, -1):                          # sons have larger ids
        nodes[k] = 1
        for s in son[k]:
            if s >= 0:
                part[k] += part[s]
                leaves[k] += leaves[s]
                nodes[k] += nodes[s]
            else:
                part[k] += T["leaf_np"][-s - 1]
                leaves[k] += 1
    big = part > 4096
    roots = [s for k in np.flatnonzero(big) for s in son[k] if s >= 0 and not big[s]]
    return len(roots), sum(bool(leaves[r] > part[r] or nodes[r] > part[r]) for r in roots)


@pytest.mark.parametrize("n,triples", [(5000, 3), (9000, 2), (40000, 8), (150000, 5)])
def test_a_subtree_that_does_not_fit(gpu_ctx, n, triples):
    g = np.random.default_rng(n)
    p = g.integers(1 << 20, 1 << 28, (n, 3))
    v = np.arange((1 << 19) + 1, (1 << 19) + 4000)
    f = v * STEP
    low = v[((f + f) + f) / 3.0 < f]                         # three of these have a mean below themselves
    for k in range(triples):
        xy = low[k * 7]
        z = int(g.integers(1 << 20, 1 << 28))
        p = np.concatenate([p, [[xy, xy, z], [xy, xy, z + 40], [xy, xy, z + 90]]])
    p = np.ascontiguousarray(p[g.permutation(len(p))], np.int32)
    tag = (g.random(len(p)) < 0.7).astype(np.int32)
    x = p.astype(np.float64) * STEP
    b = (x.min(0) - 1e-3).astype(np.float32), (x.max(0) + 1e-3).astype(np.float32)
    T = W.build_lists(p, tag, STEP, 1, np.float32(0.5), np.float32(1.0), *b, walk=False, with_tree=True)
    subtrees, misfits = _misfits(T)
    print(f"case: {len(p)} particles, {subtrees} subtrees, {misfits} that do not fit", flush=True)
    assert subtrees > misfits >= 1
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    for _ in range(2):
        nl, nn = gpu_ctx.build_tree(p, tag, STEP, 1, *b)
        dev = gpu_ctx.get_tree()
        assert (nl, nn) == (T["leaf_ip"].size, T["node_son"].shape[0])
        for k in KEYS:
            np.testing.assert_array_equal(dev[k], T[k], err_msg=k)
