"""The item queue at the sizes where its shares change: fewer items than
waves, a few per wave (the first ones dealt out), tens per wave (shares of
several items), a grid of one wave per CU; each equals the form with one wave
per item.  And the automatic item size with targets that hold no active
particle: as many items as the list of the active targets alone gives."""
import numpy as np
import pytest

import photons_p2p as pp
from photons_p2p import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def work():
    return W.uneven_pairs(seed=11, lattice=16, n_pool=900, max_src=60, reach=3, total_pairs=20000)


def _forces(ctx, w, law, exec_form, **tuning):
    ctx.set_tuning(**tuning)
    ctx.set_law(pp.ForceLaw(eps=w.eps, rs=w.rs, softening=w.softening, box=w.box, law=law))
    ctx.set_particles(w.pos, w.leaf_ip, w.leaf_np)
    ctx.set_tasks(w.task_t, w.task_s)
    ctx.compute(exec_form)
    ctx.compute(exec_form)                           # the queue starts over
    return ctx.acc(), ctx.list_stats()["nitems"]


@pytest.mark.parametrize("law", [pp.LAW_TABLE, pp.LAW_LINEAR, pp.LAW_POLY])
@pytest.mark.parametrize("waves,split", [(0, 1 << 22), (0, 1 << 15), (0, 1 << 12), (0, 1), (1, 1 << 12), (1, 1), (8, 1)])
def test_every_item_once(gpu_ctx, work, law, waves, split):
    print(f"case: law={law} waves_per_cu={waves} split={split}", flush=True)
    a, n = _forces(gpu_ctx, work, law, pp.EXEC_QUEUE, waves_per_cu=waves, split_pairs=split)
    b, m = _forces(gpu_ctx, work, law, pp.EXEC_GRID, waves_per_cu=waves, split_pairs=split)
    assert n == m
    mag = np.linalg.norm(b, axis=1)
    assert np.all(np.linalg.norm(a - b, axis=1) <= 1e-12 * np.maximum(mag, 1e-30))


@pytest.mark.parametrize("fraction", [0.5, 0.02, 0.0])
def test_automatic_size_counts_active_targets_only(gpu_ctx, work, fraction):
    g = np.random.default_rng(5)
    leaf = g.random(work.nleaf) < fraction
    act = np.repeat(leaf, work.leaf_np).astype(np.uint8)
    gpu_ctx.set_tuning()
    gpu_ctx.set_law(pp.ForceLaw(eps=work.eps, rs=work.rs, softening=work.softening, box=work.box))
    gpu_ctx.set_particles(work.pos, work.leaf_ip, work.leaf_np)
    gpu_ctx.set_active(act, 1)
    gpu_ctx.set_tasks(work.task_t, work.task_s)
    whole = gpu_ctx.list_stats()["nitems"]
    gpu_ctx.compute()
    a = gpu_ctx.acc()
    gpu_ctx.zero_acc()
    keep = leaf[work.task_t]
    gpu_ctx.set_tasks(work.task_t[keep], work.task_s[keep])
    assert gpu_ctx.list_stats()["nitems"] == whole
    gpu_ctx.compute()
    b = gpu_ctx.acc()
    assert np.all(np.abs(a - b) <= 1e-12 * np.abs(b).max(initial=1e-30))


# a list of `items` rows of one item each: fewer than workgroups, than waves (every item
# dealt, no counter), one more than either, for grids of 16 waves per CU and of one
@pytest.mark.parametrize("items", [1, 2, 255, 256, 257, 511, 512, 513, 2047, 2048, 2049, 4095, 4096, 4097, 5000])
@pytest.mark.parametrize("waves", [0, 1])
@pytest.mark.parametrize("law", [pp.LAW_TABLE, pp.LAW_LINEAR])
def test_small_lists(gpu_ctx, items, waves, law):
    print(f"case: {items} items waves_per_cu={waves} law={law}", flush=True)
    g = np.random.default_rng(items)
    nleaf = 5000
    pos = g.random((3 * nleaf, 3)) * 2.0
    gpu_ctx.set_tuning(waves_per_cu=waves)
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0, law=law))
    gpu_ctx.set_particles(pos, (3 * np.arange(nleaf)).astype(np.int32), np.full(nleaf, 3, np.int32))
    t = g.permutation(nleaf)[:items].astype(np.int32)
    gpu_ctx.set_tasks(t, g.integers(0, nleaf, items).astype(np.int32))
    out = []
    for form in (pp.EXEC_QUEUE, pp.EXEC_QUEUE, pp.EXEC_GRID):
        gpu_ctx.zero_acc()
        gpu_ctx.compute(form)
        out.append(gpu_ctx.acc())
    assert gpu_ctx.list_stats()["nitems"] == items
    # the same items, each by one wave: equal to the bit
    assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[2])


# rows about the 16 lanes that search a cut together (one probe each, a second
# round, a partial last round): as many items as a scan of each row cuts
@pytest.mark.parametrize("sources", [1, 2, 15, 16, 17, 18, 255, 256, 257, 273, 290, 4097])
@pytest.mark.parametrize("split", [1, 700, 9000, 300000])
def test_cuts_of_a_row(gpu_ctx, sources, split):
    print(f"case: {sources} sources split={split}", flush=True)
    g = np.random.default_rng(sources)
    num = g.integers(1, 9, 300).astype(np.int32)
    num[7], num[8] = 5, 200                                  # the targets: one chunk, and two
    ip = (np.cumsum(num) - num).astype(np.int32)
    gpu_ctx.set_tuning(split_pairs=split)
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(g.random((int(num.sum()), 3)), ip, num)
    s = np.stack([g.integers(0, 300, sources) for _ in range(2)]).astype(np.int32)
    gpu_ctx.set_tasks(np.repeat(np.array([7, 8], np.int32), sources), s.reshape(-1))
    expect = 0
    for ni, src in ((5, s[0]), (200, s[1])):
        chunks = (ni + 191) // 192
        wi = (ni + chunks - 1) // chunks + 24                # the staging counts as 24 pairs
        run, ranges = 0, 1
        for n in num[src]:
            if run and (run + int(n)) * wi > split:
                ranges, run = ranges + 1, 0
            run += int(n)
        expect += ranges * chunks
    assert gpu_ctx.list_stats()["nitems"] == expect
    gpu_ctx.set_tuning()


# item counts about a workgroup of the cost sort (1024 items) with costs over many
# classes: every item once in the sorted copy, so that both copies give the same
# sums (one item per target: equal to the bit)
@pytest.mark.parametrize("items", [1, 1023, 1024, 1025, 2049, 9000])
def test_sorted_items(gpu_ctx, items):
    print(f"case: {items} items", flush=True)
    g = np.random.default_rng(items)
    num = (10 ** (2.2 * g.random(9000))).astype(np.int32)    # 1 to 158 particles
    gpu_ctx.set_tuning(split_pairs=1 << 30)
    gpu_ctx.set_law(pp.ForceLaw(eps=0.05, rs=1.0))
    gpu_ctx.set_particles(g.random((int(num.sum()), 3)), (np.cumsum(num) - num).astype(np.int32), num)
    t = g.permutation(9000)[:items].astype(np.int32)
    gpu_ctx.set_tasks(np.repeat(t, 3), g.integers(0, 9000, 3 * items).astype(np.int32))
    out = []
    for form in (pp.EXEC_QUEUE, pp.EXEC_GRID):
        gpu_ctx.zero_acc()
        gpu_ctx.compute(form)
        out.append(gpu_ctx.acc())
    assert gpu_ctx.list_stats()["nitems"] == items
    assert np.array_equal(out[0], out[1])
    gpu_ctx.set_tuning()
