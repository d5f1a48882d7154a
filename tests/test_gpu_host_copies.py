"""Copies between host arrays and the device at the sizes where their form
changes (4 MiB, pieces of up to 2 MiB, slices of 128 KiB, a last odd piece): lists
come back as they went, positions from plain arrays and from 40-byte records
reach every particle, and a bad leaf id anywhere in a long list is refused."""
import numpy as np
import pytest

import photons_p2p as pp

pytestmark = pytest.mark.gpu

SIZES = [1, 5000, 1048575, 1048576, 1048577, 2097152, 2097153, 3 * 1048576 + 65537, 5 * 1048576 - 1]


def _context(ctx, n, nleaf=7):
    ip = (np.arange(nleaf) * n // nleaf).astype(np.int32)
    num = np.diff(np.append(ip, n)).astype(np.int32)
    ctx.set_tuning()
    ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    return ip, num


@pytest.mark.parametrize("n", SIZES)
def test_lists_round_trip(gpu_ctx, n):
    print(f"case: list of {n}", flush=True)
    ip, num = _context(gpu_ctx, 70)
    gpu_ctx.set_particles(np.random.default_rng(0).random((70, 3)), ip, num)
    g = np.random.default_rng(n)
    t, s = g.integers(0, 7, n).astype(np.int32), g.integers(0, 7, n).astype(np.int32)
    gpu_ctx.set_tasks(t, s)
    gpu_ctx.add_tasks(s[: n // 3], t[: n // 3])
    tt, ts = gpu_ctx.get_tasks()
    assert np.array_equal(tt, np.concatenate([t, s[: n // 3]])) and np.array_equal(ts, np.concatenate([s, t[: n // 3]]))
    bad = t.copy()
    bad[2 * n // 3] = 7
    with pytest.raises(pp.P2PError, match=f"task {2 * n // 3} "):
        gpu_ctx.add_tasks(s, bad)
    assert gpu_ctx.get_tasks()[0].size == n + n // 3         # the list is as it was
    bad[2 * n // 3] = -1
    with pytest.raises(pp.P2PError, match=f"task {2 * n // 3} "):
        gpu_ctx.set_tasks(bad, s)


@pytest.mark.parametrize("n", [7, 3000, 43690, 87381, 87382, 349525, 349526, 700001])
def test_positions_reach_every_particle(gpu_ctx, n):
    """A local expansion whose force is the position itself (L_xx = L_yy =
    L_zz = 1 about the origin) returns every particle's FP32 position."""
    print(f"case: {n} particles", flush=True)
    ip, num = _context(gpu_ctx, n)
    g = np.random.default_rng(n)
    L = np.zeros((7, 20), np.float32)
    L[:, [4, 7, 9]] = 1.0
    zero = np.zeros((7, 3), np.float32)
    posi = g.integers(-(1 << 28), 1 << 30, (n, 3)).astype(np.int32)
    rec = np.zeros(n, dtype=[("posi", np.int32, 3), ("rest", np.int32, 7)])
    rec["posi"], rec["rest"] = posi, 77
    x = posi.astype(np.float64) * 1.7e-7
    for put in (lambda: gpu_ctx.set_particles(x, ip, num), lambda: gpu_ctx.set_particles_i32(posi, 1.7e-7, ip, num),
                lambda: gpu_ctx.set_particles_i32(rec, 1.7e-7, ip, num)):
        put()
        gpu_ctx.l2p(L, zero)
        want = x.astype(np.float32)
        assert np.array_equal(gpu_ctx.acc(), want.astype(np.float64))
        assert np.array_equal(gpu_ctx.acc_f32_soa(), want.T)


def test_leaves_out_of_order(gpu_ctx):
    """Ranges that do not ascend are accepted when disjoint, refused when not."""
    ip, num = np.array([40, 0, 10, 10], np.int32), np.array([30, 10, 0, 30], np.int32)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    x = np.random.default_rng(1).random((70, 3))
    gpu_ctx.set_particles(x, ip, num)
    for bad in ([39, 0, 10, 10], [40, 0, 10, 11]):
        with pytest.raises(pp.P2PError):
            gpu_ctx.set_particles(x, np.array(bad, np.int32), num)
