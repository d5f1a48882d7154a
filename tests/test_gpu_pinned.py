"""Arrays in pinned host memory, copied straight from 4 MiB on: positions, lists
and results of a context equal those of ordinary arrays, a bad leaf id is
refused, an array that only begins in pinned memory works; and the drop-in
library, which keeps its lists and results pinned, with flushes of more than 4 MiB."""
import ctypes

import numpy as np
import pytest

import photons_p2p as pp
from photons_p2p import workloads as W
from test_gpu_dropin import Host, libs  # noqa: F401
from test_zz_no_alloc import _hip_lib

pytestmark = pytest.mark.gpu


class Pinned:
    """Pinned copies of numpy arrays."""

    def __init__(self):
        self.ptrs = []

    def __call__(self, a):
        a = np.ascontiguousarray(a)
        p = ctypes.c_void_p()
        h = _hip_lib()
        h.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
        h.hipHostFree.argtypes = [ctypes.c_void_p]
        assert h.hipHostMalloc(ctypes.byref(p), a.nbytes, 0) == 0
        self.ptrs.append(p)
        b = np.frombuffer((ctypes.c_char * a.nbytes).from_address(p.value), a.dtype).reshape(a.shape)
        b[:] = a
        return b

    def free(self):
        for p in self.ptrs:
            _hip_lib().hipHostFree(p)


@pytest.fixture()
def pinned():
    p = Pinned()
    yield p
    p.free()


def test_context_arrays(gpu_ctx, pinned):
    g = np.random.default_rng(2)
    n, nleaf, ntask = 400001, 20000, 1400003
    ip = (np.arange(nleaf) * n // nleaf).astype(np.int32)
    num = np.diff(np.append(ip, n)).astype(np.int32)
    x = g.random((n, 3)) * 40
    posi = g.integers(0, 1 << 28, (n, 3)).astype(np.int32)
    t, s = g.integers(0, nleaf, ntask).astype(np.int32), g.integers(0, nleaf, ntask).astype(np.int32)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    zero = np.zeros((nleaf, 3), np.float32)
    L = np.zeros((nleaf, 20), np.float32)
    L[:, [4, 7, 9]] = 1.0                                    # the force is the position
    print("case: positions", flush=True)
    for put, want in ((lambda: gpu_ctx.set_particles(pinned(x), ip, num), x),
                      (lambda: gpu_ctx.set_particles_i32(pinned(posi), 1.7e-7, ip, num), posi.astype(np.float64) * 1.7e-7)):
        put()
        gpu_ctx.l2p(pinned(L), zero)
        assert np.array_equal(gpu_ctx.acc(), want.astype(np.float32).astype(np.float64))
        out = pinned(np.zeros((3, n), np.float32))
        gpu_ctx._chk(gpu_ctx._lib.pp2p_get_acc_f32_soa(gpu_ctx._h, out.ctypes.data))
        assert np.array_equal(out, want.astype(np.float32).T)
    print("case: lists", flush=True)
    tp, sp = pinned(t), pinned(s)
    gpu_ctx.set_tasks(tp, sp)
    gpu_ctx.add_tasks(s, tp)                                 # one pinned, one not
    tt, ts = gpu_ctx.get_tasks()
    assert np.array_equal(tt, np.concatenate([t, s])) and np.array_equal(ts, np.concatenate([s, t]))
    for k in (0, ntask // 2, ntask - 1):
        tp[k] = nleaf
        with pytest.raises(pp.P2PError, match=f"task {k} "):
            gpu_ctx.add_tasks(s, tp)
        tp[k] = t[k]
    assert gpu_ctx.get_tasks()[0].size == 2 * ntask


def test_long_flushes_through_the_dropin(gpu_ctx, libs):  # noqa: F811
    """Each flush waited for, so that it is one list: the same items as that list
    in a context, whose FP64 sums differ by their order alone."""
    host, lib = libs
    w = W.config_plain(72, softening=0)
    H = Host(host, w)
    nt, len_task = w.task_t.size, 1300000
    assert 12 * w.npart >= 4 << 20 and nt > 2 * len_task
    flushes = [slice(k, min(k + len_task, nt)) for k in range(0, nt, len_task)]
    gpu_ctx.set_tuning()
    f32 = lambda v: float(np.float32(v))  # noqa: E731     the host program's scales are floats
    gpu_ctx.set_law(pp.ForceLaw(eps=f32(w.eps), rs=f32(w.rs), softening=pp.SOFT_REF))
    gpu_ctx.set_particles_i32(w.meta["posi"], w.meta["int2pos"], w.leaf_ip, w.leaf_np)
    for f in flushes:
        gpu_ctx.set_tasks(w.task_t[f], w.task_s[f])
        gpu_ctx.compute()
    want = gpu_ctx.acc_f32_soa()
    assert np.abs(want).max() > 0
    lib.hostmalloc_task(len_task)
    pt, ps = H.tasks()
    tt, ts = (np.ctypeslib.as_array(p, (len_task,)) for p in (pt, ps))
    for step in range(2):                                    # the second step finds its buffers pinned
        print(f"case: drop-in step {step}, {nt} tasks in flushes of {len_task}", flush=True)
        for a in H.acc:
            a[:] = 0.0
        ctypes.c_int.in_dll(host, "NPACK").value = 0
        for f in flushes:
            n = f.stop - f.start
            tt[:n] = w.task_t[f] + H.first_leaf
            ts[:n] = w.task_s[f] + H.first_leaf
            lib.task_compute_p2p_gpu(n, pt, ps, int(f.stop == nt))
            assert lib.p2p_hip_status() == 0, lib.p2p_hip_error()       # waits for the flush
        lib.hostmalloc_out(w.npart)
        lib.devMemcpyDH_updateAcc(H.packs, H.npack(), -1)
        lib.hostfree_out()
        assert lib.p2p_hip_status() == 0, lib.p2p_hip_error()
        got = np.stack(H.acc)
        d = np.abs(got - want)
        print(f"largest difference {d.max():.2e} of {np.abs(want).max():.2e}", flush=True)
        assert np.all(d <= 2.0 ** -22 * np.abs(want) + 1e-9 * np.abs(want).max())
    lib.hostfree_task()
