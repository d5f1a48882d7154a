"""Targets of more i-chunks than the 16 lanes that emit a row's items (a lane
then writes several of them), with one and with several source ranges: as many
items as the rule gives, and forces that the FP64 oracle gives, so that no
chunk is missing or written twice."""
import numpy as np
import pytest

import photons_p2p as pp
import pyoracle

pytestmark = pytest.mark.gpu


# 16 chunks of 192 (the last one-lane emission), 17, 33; and small chunks of a moderate leaf
@pytest.mark.parametrize("target,chunk", [(3072, 0), (3073, 0), (6200, 0), (200, 5), (160, 10), (170, 10), (333, 10)])
@pytest.mark.parametrize("split", [1 << 30, 40000, 1])
def test_chunks_past_the_lanes(gpu_ctx, target, chunk, split):
    print(f"case: target of {target} chunk_model={chunk} split={split}", flush=True)
    g = np.random.default_rng(target + chunk)
    num = g.integers(1, 9, 60).astype(np.int32)
    num[7] = target
    ip = (np.cumsum(num) - num).astype(np.int32)
    x = g.random((int(num.sum()), 3)) * 2.0
    t = np.concatenate([np.full(40, 7), [3, 3, 9]]).astype(np.int32)
    s = np.concatenate([g.permutation(60)[:40], [7, 1, 2]]).astype(np.int32)
    s[:40][s[:40] == 7] = 6
    gpu_ctx.set_tuning(split_pairs=split, chunk_model=chunk)
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(x, ip, num)
    gpu_ctx.set_tasks(t, s)
    expect = 0
    for tgt in (3, 7, 9):
        src, ni = s[t == tgt], int(num[tgt])
        cap = min(chunk, 192) if chunk > 0 else 192
        k = -(-ni // cap)
        wi = -(-ni // k) + 24                                # the staging counts as 24 pairs
        run, ranges = 0, 1
        for n in num[src]:
            if run and (run + int(n)) * wi > split:
                ranges, run = ranges + 1, 0
            run += int(n)
        expect += ranges * k
    assert gpu_ctx.list_stats()["nitems"] == expect
    ref = pyoracle.p2p_f64(pyoracle.params(0.05, 1.0, softening=0), x, ip, num, pyoracle.build_csr(t, s, 60))
    for form in (pp.EXEC_QUEUE, pp.EXEC_GRID):
        gpu_ctx.zero_acc()
        gpu_ctx.compute(form)
        a = gpu_ctx.acc()
        # pair forces of FP32 (a few 1e-7 each); a missing or doubled chunk is off by its whole force
        assert np.abs(a - ref).max() <= 1e-5 * np.abs(ref).max()
        assert np.all((np.abs(a).max(1) > 0) == (np.abs(ref).max(1) > 0))
    gpu_ctx.set_tuning()
