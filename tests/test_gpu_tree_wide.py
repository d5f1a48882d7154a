"""The device tree where a level holds more segments than a grid has workgroups
in one dimension (2^22 of 1024 threads): pairs of particles on a lattice of 2^22 sites in
leaves of one, with one empty leaf (three equal coordinates whose rounded mean
lies below them), so that a subtree has more leaves than particles and every
level runs over the device.  Array for array against the host builder."""
import numpy as np
import pytest

import photons_p2p as pp
from photons_p2p import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("perm", "leaf_ip", "leaf_np", "active", "leaf_center", "leaf_width", "node_son", "node_center", "node_width")


def test_more_segments_than_a_grid_row():
    step = 1.7e-7
    g = np.random.default_rng(0)
    q = np.stack(np.meshgrid(np.arange(256) << 20, np.arange(128) << 21, np.arange(128) << 21, indexing="ij"), -1)
    q = q.reshape(-1, 3) + (1 << 19)
    p = np.concatenate([q, q + g.integers(1, 900, q.shape)])
    v = np.arange(1, 4000) + int(q[77, 1])
    f = v * step
    y = int(v[((f + f) + f) / 3.0 < f][0])
    p[77] = q[77, 0], y, q[77, 2]
    p[77 + len(q)] = q[77, 0] + 5, y, q[77, 2] + 300
    p = np.concatenate([p, [[q[77, 0] + 9, y, q[77, 2] + 700]]])
    p = np.ascontiguousarray(p[g.permutation(len(p))], np.int32)
    tag = (g.random(len(p)) < 0.7).astype(np.int32)
    x = p.astype(np.float64) * step
    b = (x.min(0) - 1e-3).astype(np.float32), (x.max(0) + 1e-3).astype(np.float32)
    host = W.build_lists(p, tag, step, 1, np.float32(0.5), np.float32(1.0), *b, walk=False, with_tree=True)
    assert np.sum(host["leaf_np"] == 0) == 1
    level = np.array([0])
    widest = 0
    while level.size:
        widest = max(widest, level.size)
        son = host["node_son"][level].ravel()
        level = son[son >= 0]
    assert widest == 1 << 22
    print(f"case: {len(p)} particles, {widest} segments on a level", flush=True)
    with pp.Context(0) as ctx:                       # its 10 GB go with it
        ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
        nl, nn = ctx.build_tree(p, tag, step, 1, *b)
        assert (nl, nn) == (host["leaf_ip"].size, host["node_son"].shape[0])
        dev = ctx.get_tree()
    for k in KEYS:
        assert np.array_equal(dev[k], host[k]), k
