"""Arrays that reach the host through the pinned mailbox, at the sizes where one
workgroup, several, two mails or a copy take them (8192 words, 512 KiB): lists
come back as they went, and accelerations are the FP64 ones rounded once."""
import numpy as np
import pytest

import photons_p2p as pp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4096, 4097, 8191, 8193, 65535, 65536, 65537, 131071, 131072, 131073])
def test_lists_by_mail(gpu_ctx, n):
    print(f"case: list of {n}", flush=True)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    ip = (np.arange(7) * 10).astype(np.int32)
    gpu_ctx.set_particles(np.random.default_rng(0).random((70, 3)), ip, np.full(7, 10, np.int32))
    g = np.random.default_rng(n)
    for _ in range(2):                                       # the second mail is not the first one's
        t, s = g.integers(0, 7, n).astype(np.int32), g.integers(0, 7, n).astype(np.int32)
        gpu_ctx.set_tasks(t, s)
        tt, ts = gpu_ctx.get_tasks()
        assert np.array_equal(tt, t) and np.array_equal(ts, s)


@pytest.mark.parametrize("n", [1, 2730, 2731, 43690, 43691, 50000])
def test_accelerations_by_mail(gpu_ctx, n):
    print(f"case: {n} particles", flush=True)
    g = np.random.default_rng(n)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(g.random((n, 3)) * 30, np.zeros(1, np.int32), np.full(1, n, np.int32))
    L = g.standard_normal((1, 20)).astype(np.float32)
    gpu_ctx.zero_acc()
    gpu_ctx.l2p(L, np.full((1, 3), 15.0, np.float32))
    a64, a32 = gpu_ctx.acc(), gpu_ctx.acc_f32_soa()
    assert np.abs(a64).max() > 0
    assert np.array_equal(a32, a64.T.astype(np.float32))
