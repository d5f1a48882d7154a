"""The work that programs have this library do, as measurable cases.

A cosmological N-body program calls the library in a few ways, and the cases
cover each from the smallest box to a large one:

  step       a whole force evaluation from grid positions, all on the device:
             tree, walk, short-range pairs, multipoles and particle mesh, then
             the accelerations and the tree's particle order back on the host
  tree       the kd-tree and the interaction list alone, fetched by a program
             that evaluates or schedules the lists itself
  force      one evaluation over a list that stays on the device
  active     the same for the particles of one time-step level (a new mask
             each sub-step)
  hostlists  the reference's own protocol: 40-byte particle records and a
             leaf-pair list arrive from host code, the forces go back
  uneven     leaf pairs of very different sizes in a periodic box
  multipole  the M2L task loop and L2P of a program with its own tree
  mesh       the long-range particle-mesh force alone

Particles are drawn on the GPU from the seed: a Zel'dovich-displaced grid
("plain"), or half of one and half in Plummer spheres ("clustered"), the two
distributions of the repository's benchmark, with periodic ghost copies
within the cutoff as a domain imports them.  Force-law scales follow the
reference: split radius 1.25 mesh cells, tree cutoff 4.5 split radii,
softening 0.03 cells (REF) or spacing / 40 (Plummer).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "photons-on-mt3000_amd"))

import photons_p2p as pp  # noqa: E402

UCUT = 2.8125
BOX = 100.0          # box length of the tree-based cases
MASS = 0.37
GPU = torch.device("cuda")


# --------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest whole step (a test problem, or one small domain): launches and synchronisations
        {"name": "step_16", "kind": "step", "n1": 16, "dist": "plain", "maxleaf": 32, "theta": 0.5, "law": "table", "soft": "plummer"},
        # the plain benchmark configuration, every part of the force
        {"name": "step_64", "kind": "step", "n1": 64, "dist": "plain", "maxleaf": 32, "theta": 0.5, "law": "table", "soft": "ref"},
        # the benchmark's clustered box at its size: the production step of one GPU
        {"name": "step_256_clustered", "kind": "step", "n1": 256, "dist": "clustered", "maxleaf": 64, "theta": 0.5, "law": "linear", "soft": "plummer"},
        # lists for host code: tree and walk, every array fetched (an odd number of particles)
        {"name": "tree_111_clustered", "kind": "tree", "n1": 111, "dist": "clustered", "maxleaf": 64, "theta": 0.5},
        # a sub-domain's resident list, evaluated again and again: latency
        {"name": "force_12", "kind": "force", "n1": 12, "dist": "plain", "maxleaf": 32, "theta": 0.5, "law": "table", "soft": "ref"},
        # the plain benchmark list, the default law
        {"name": "force_64", "kind": "force", "n1": 64, "dist": "plain", "maxleaf": 32, "theta": 0.5, "law": "table", "soft": "plummer"},
        # a clustered list of many long rows, the linear law
        {"name": "force_144_clustered", "kind": "force", "n1": 144, "dist": "clustered", "maxleaf": 64, "theta": 0.5, "law": "linear", "soft": "plummer"},
        # one deep time-step level: 5% of the particles
        {"name": "active_96_clustered", "kind": "active", "n1": 96, "dist": "clustered", "maxleaf": 64, "theta": 0.5, "law": "linear", "soft": "plummer", "fraction": 0.05},
        # particle records and lists from the host every step, odd and ragged
        {"name": "hostlists_75_clustered", "kind": "hostlists", "n1": 75, "dist": "clustered", "maxleaf": 48, "theta": 0.5, "law": "table", "soft": "ref"},
        # the uneven batching workload: leaves of 1 to 256 particles, 1 to 400 sources
        {"name": "uneven_1m", "kind": "uneven", "lattice": 64, "pairs": 1000000, "law": "linear", "soft": "plummer"},
        # M2L and L2P for a program with its own tree
        {"name": "multipole_48", "kind": "multipole", "n1": 48, "dist": "clustered", "maxleaf": 8, "theta": 0.7},
        # the mesh force of one domain: local particles and ghosts told apart by tags
        {"name": "mesh_100", "kind": "mesh", "n1": 100, "dist": "clustered", "mesh": 128, "tags": True},
    ]


def draw(rng):
    kind = rng.choice(["step", "step", "tree", "force", "force", "active", "hostlists", "uneven", "multipole", "mesh"])
    top = {"step": 160, "tree": 128, "force": 128, "active": 112, "hostlists": 96, "multipole": 56, "mesh": 128}
    if kind == "uneven":
        return {"kind": kind, "lattice": rng.choice([24, 40, 64]), "pairs": int(math.exp(rng.uniform(math.log(2e4), math.log(1e6)))),
                "law": rng.choice(["table", "linear"]), "soft": rng.choice(["ref", "plummer"])}
    n1 = int(math.exp(rng.uniform(math.log(11), math.log(top[kind]))))
    c = {"kind": kind, "n1": n1, "dist": rng.choice(["plain", "clustered"])}
    if kind == "mesh":
        c.update(mesh=2 * int(rng.uniform(0.4, 0.7) * n1 + 4), tags=rng.random() < 0.5)
        return c
    c.update(maxleaf=rng.randrange(6, 16) if kind == "multipole" else rng.randrange(32 if kind == "tree" else 16, 80),
             theta=round(rng.uniform(0.4, 0.7), 2))
    if kind not in ("tree", "multipole"):
        c.update(law=rng.choice(["table", "linear"]), soft=rng.choice(["ref", "plummer"]))
    if kind == "active":
        c["fraction"] = round(math.exp(rng.uniform(math.log(0.01), math.log(0.5))), 3)
    return c


# -------------------------------------------------------------------- inputs

def generator(seed):
    return torch.Generator(device=GPU).manual_seed(int(seed))


def zeldovich(n, box, g):
    """n^3 grid displaced by a Gaussian field with P(k) ~ k^-2, rms 0.3 spacings."""
    w = torch.fft.rfftn(torch.randn(n, n, n, generator=g, device=GPU))
    k = torch.fft.fftfreq(n, device=GPU)
    ks = (k[:, None, None], k[None, :, None], torch.fft.rfftfreq(n, device=GPU)[None, None, :])
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    k2[0, 0, 0] = 1.0
    amp = k2 ** -1.5
    amp[0, 0, 0] = 0.0
    psi = torch.stack([torch.fft.irfftn(1j * q * amp * w, s=(n, n, n)).reshape(-1) for q in ks], 1).double()
    d = box / n
    psi *= 0.3 * d / psi.square().sum(1).mean().sqrt()
    a = (torch.arange(n, device=GPU, dtype=torch.float64) + 0.5) * d
    grid = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    return (grid + psi) % box


def plummer(total, box, spacing, g):
    """Plummer spheres of masses over three decades, one per ~8000 particles."""
    m = max(8, total // 4000)
    mass = 10.0 ** (3.0 * torch.rand(m, generator=g, device=GPU, dtype=torch.float64))
    owner = torch.searchsorted(mass.cumsum(0), torch.rand(total, generator=g, device=GPU, dtype=torch.float64) * mass.sum()).clamp_max(m - 1)
    centre = torch.rand(m, 3, generator=g, device=GPU, dtype=torch.float64) * box
    a = (0.5 + 4.5 * torch.rand(m, generator=g, device=GPU, dtype=torch.float64)) * spacing
    x = torch.rand(total, generator=g, device=GPU, dtype=torch.float64).clamp_min(1e-12) * (1000.0 / 101.0 ** 1.5)
    r = a[owner] / (x ** (-2.0 / 3.0) - 1.0).sqrt()
    v = torch.randn(total, 3, generator=g, device=GPU, dtype=torch.float64)
    return (centre[owner] + r[:, None] * v / v.norm(dim=1, keepdim=True)) % box


def scales(case):
    """Split radius, tree cutoff, grid step and softening of a tree-based case."""
    cell = BOX / case["n1"]
    rs = 1.25 * cell
    cutoff = 4.5 * rs
    eps = cell / 40.0 if case.get("soft") == "plummer" else 0.03 * cell
    return rs, cutoff, (BOX + cutoff * 1.1) / (1 << 30), eps


def particles(case, seed):
    """Integer grid positions (local particles, then ghost copies) and tags, on the GPU."""
    g = generator(seed)
    n1 = case["n1"]
    pos = zeldovich(n1, BOX, g)
    if case["dist"] == "clustered":
        n = pos.shape[0]
        keep = torch.rand(n, generator=g, device=GPU) < 0.5
        pos = torch.cat([pos[keep], plummer(n - int(keep.sum()), BOX, BOX / n1, g)])
    _, cutoff, step, _ = scales(case)
    box_i = int(round(BOX / step))
    p = torch.floor(pos / step).long() % box_i
    if case["kind"] == "multipole":                  # an isolated box
        return p.int(), torch.ones(p.shape[0], dtype=torch.int32, device=GPU)
    # the closest copies: as many as a shell of the cutoff's width holds on average
    count = int(p.shape[0] * ((1.0 + 2.0 * cutoff / BOX) ** 3 - 1.0))
    width = math.ceil(1.2 * cutoff / step)
    while True:
        every = p
        for d in range(3):                           # images axis by axis: corners come from the earlier axes' copies
            lo = every[every[:, d] < width].clone()
            hi = every[every[:, d] >= box_i - width].clone()
            lo[:, d] += box_i
            hi[:, d] -= box_i
            every = torch.cat([every, lo, hi])
        ghosts = every[p.shape[0]:]
        if ghosts.shape[0] >= count:
            break
        width = min(box_i, int(1.3 * width))
    far = torch.maximum(-ghosts, ghosts - (box_i - 1)).amax(1)
    near = torch.sort(torch.argsort(far, stable=True)[:count]).values
    posi = torch.cat([p, ghosts[near]])
    tag = torch.zeros(posi.shape[0], dtype=torch.int32, device=GPU)
    tag[:p.shape[0]] = 1
    return posi.int(), tag


def bounds(posi, step):
    """Root box: FP32 positions widened by 1e-6 of the box length."""
    x = (posi.double() * step).float()
    lo, hi = x.amin(0).cpu().numpy(), x.amax(0).cpu().numpy()
    return ((np.minimum(lo, BOX) - 1e-6 * BOX).astype(np.float32), (np.maximum(hi, 0) + 1e-6 * BOX).astype(np.float32))


def kdtree(posi, tag, step, maxleaf):
    """Mean-split kd-tree, level by level: particle order, leaf ranges, cell
    boxes (centre, width; leaves first, then nodes), sons and local leaves."""
    n = posi.shape[0]
    order = torch.arange(n, device=GPU)
    lo_b, hi_b = bounds(posi, step)
    start, size = torch.zeros(1, dtype=torch.long, device=GPU), torch.full((1,), n, device=GPU)
    lo, hi = torch.tensor(lo_b, device=GPU)[None], torch.tensor(hi_b, device=GPU)[None]
    node_box, sons, leaves = [], [], []              # sons: (level, child slot) resolved at the end
    nnode, nleaf, axis = 0, 0, 0
    while start.numel():
        m = start.numel()
        node_box.append((lo, hi))
        seg = torch.repeat_interleave(torch.arange(m, device=GPU), size)
        first = size.cumsum(0) - size
        at = start[seg] + torch.arange(seg.numel(), device=GPU) - first[seg]
        x = posi[order[at], axis].long()
        mean = torch.zeros(m, dtype=torch.long, device=GPU).index_add_(0, seg, x).double() / size
        small = x.double() <= mean[seg]
        c = torch.cat([torch.zeros(1, dtype=torch.long, device=GPU), small.long().cumsum(0)])
        left = c[first + size] - c[first]
        last = torch.arange(seg.numel(), device=GPU) == (first + size - 1)[seg]
        small &= ~(last & (left == size)[seg])       # coincident particles: the last one goes right
        c = torch.cat([torch.zeros(1, dtype=torch.long, device=GPU), small.long().cumsum(0)])
        left = c[first + size] - c[first]
        rank = c[:-1] - c[first][seg]
        off = torch.arange(seg.numel(), device=GPU) - first[seg]
        to = start[seg] + torch.where(small, rank, left[seg] + off - rank)
        order[to] = order[at].clone()
        split = (mean * step).float()
        cs = torch.stack([start, start + left], 1).reshape(-1)
        cn = torch.stack([left, size - left], 1).reshape(-1)
        clo, chi = lo.repeat_interleave(2, 0), hi.repeat_interleave(2, 0)
        chi[0::2, axis] = split
        clo[1::2, axis] = split
        isn = cn > maxleaf
        ids = torch.empty_like(cs)
        ids[isn] = nnode + m + torch.arange(int(isn.sum()), device=GPU)
        ids[~isn] = -1 - (nleaf + torch.arange(int((~isn).sum()), device=GPU))
        sons.append(ids.reshape(-1, 2))
        leaves.append((cs[~isn], cn[~isn], clo[~isn], chi[~isn]))
        nnode, nleaf = nnode + m, nleaf + int((~isn).sum())
        start, size, lo, hi = cs[isn], cn[isn], clo[isn], chi[isn]
        axis = (axis + 1) % 3
    ip, num, llo, lhi = (torch.cat(v) for v in zip(*leaves))
    by = torch.argsort(ip * 2 + (num > 0))           # leaves in particle order
    new = torch.empty_like(by)
    new[by] = torch.arange(nleaf, device=GPU)
    sons = torch.cat(sons)
    sons = torch.where(sons < 0, -1 - new[(-1 - sons).clamp_min(0)], sons)
    nlo, nhi = (torch.cat(v) for v in zip(*node_box))
    lo, hi = torch.cat([llo[by], nlo]), torch.cat([lhi[by], nhi])
    ip, num = ip[by], num[by]
    c = torch.cat([torch.zeros(1, dtype=torch.long, device=GPU), (tag[order] == 1).long().cumsum(0)])
    return {"order": order, "ip": ip, "np": num, "center": 0.5 * (lo + hi), "width": hi - lo, "sons": sons,
            "local": c[ip + num] > c[ip]}


def median_tree(posi, step, maxleaf):
    """Median-split tree with tight boxes: the same fields as kdtree()."""
    n = posi.shape[0]
    levels = max(1, math.ceil(math.log2(n / maxleaf)))
    order, size = torch.arange(n, device=GPU), torch.full((1,), n, device=GPU)
    for level in range(levels):
        seg = torch.repeat_interleave(torch.arange(size.numel(), device=GPU), size)
        order = order[torch.argsort((seg << 32) + (posi[order, level % 3].long() + (1 << 30)), stable=True)]
        size = torch.stack([size // 2, size - size // 2], 1).reshape(-1)
    leaf = torch.repeat_interleave(torch.arange(size.numel(), device=GPU), size)[:, None].expand(n, 3)
    x = (posi[order].double() * step).float()
    lo = torch.zeros(size.numel(), 3, device=GPU).scatter_reduce_(0, leaf, x, "amin", include_self=False)
    hi = torch.zeros(size.numel(), 3, device=GPU).scatter_reduce_(0, leaf, x, "amax", include_self=False)
    boxes = [(lo, hi)]
    for _ in range(levels):
        boxes.insert(0, (torch.minimum(boxes[0][0][0::2], boxes[0][0][1::2]), torch.maximum(boxes[0][1][0::2], boxes[0][1][1::2])))
    lo, hi = (torch.cat([v[-1], *v[:-1]]) for v in zip(*boxes))
    nnode = size.numel() - 1
    sons = 1 + torch.arange(2 * nnode, device=GPU)
    sons = torch.where(sons < nnode, sons, -1 - (sons - nnode)).reshape(-1, 2)
    return {"order": order, "ip": size.cumsum(0) - size, "np": size, "center": 0.5 * (lo + hi), "width": hi - lo, "sons": sons,
            "local": torch.ones(size.numel(), dtype=torch.bool, device=GPU)}


def interleave(t, s, bits):
    """Z-order key of the pair: for one target the sources ascend, as in the order of a depth-first dual walk."""
    key = torch.zeros_like(t)
    for b in range(bits):
        key |= ((t >> b) & 1) << (2 * b + 1) | ((s >> b) & 1) << (2 * b)
    return key


def dual_walk(tree, theta, cutoff):
    """Leaf pairs within the cutoff that must be summed directly, and the
    well-separated cell pairs (cells: leaf id, or leaves + node id)."""
    nl = tree["ip"].numel()
    c, w = tree["center"], tree["width"]
    sons = torch.where(tree["sons"] < 0, -1 - tree["sons"], nl + tree["sons"])
    a = b = torch.full((1,), nl, dtype=torch.long, device=GPU)
    if sons.numel() == 0:
        raise ValueError("the tree has one leaf only")
    pt, ps, mt, ms = [], [], [], []
    wsum = w.sum(1)
    while a.numel():
        half = 0.5 * (w[a] + w[b])
        d = c[a] - c[b]
        gap = (d.abs() - half).clamp_min(0)
        touch = (gap.sum(1) <= 0) | (a == b)
        near = touch | (gap.square().sum(1) <= cutoff * cutoff)
        sep = near & ~touch & ((2 * half.amax(1)) ** 2 < theta * theta * d.square().sum(1))
        both = (a < nl) & (b < nl)
        take = both & tree["local"][a.clamp_max(nl - 1)]     # every leaf pair reached is listed, as the reference's walk does
        pt.append(a[take])
        ps.append(b[take])
        mt.append(a[sep & ~both])
        ms.append(b[sep & ~both])
        go = near & ~sep & ~both
        a, b = a[go], b[go]
        same = a == b
        x, y = sons[a[same] - nl, 0], sons[a[same] - nl, 1]
        ta = ~same & (a >= nl) & ((b < nl) | (wsum[a] > wsum[b]))
        tb = ~same & ~ta
        xa, ya = sons[a[ta] - nl, 0], sons[a[ta] - nl, 1]
        xb, yb = sons[b[tb] - nl, 0], sons[b[tb] - nl, 1]
        a, b = (torch.cat([x, x, y, y, xa, ya, a[tb], a[tb]]), torch.cat([x, y, x, y, b[ta], b[ta], xb, yb]))
    t, s = torch.cat(pt), torch.cat(ps)
    by = torch.argsort(interleave(t, s, max(1, (nl - 1).bit_length())))
    return t[by], s[by], torch.cat(mt), torch.cat(ms)


def tree_list(case, seed):
    """Tree-ordered grid positions, leaves and the leaf-pair list of a case."""
    posi, tag = particles(case, seed)
    _, cutoff, step, _ = scales(case)
    tree = median_tree(posi, step, case["maxleaf"]) if case["kind"] == "multipole" else kdtree(posi, tag, step, case["maxleaf"])
    t, s, mt, ms = dual_walk(tree, case["theta"], cutoff)
    return {"posi": posi[tree["order"]], "tag": tag[tree["order"]], "ip": tree["ip"], "np": tree["np"], "t": t, "s": s,
            "mt": mt, "ms": ms, "tree": tree}


def active_levels(case, seed, inp):
    """uint8 levels: `fraction` of the local particles, whole clumps first (neighbours in tree order), are at level 1."""
    g = generator(seed + 7919)
    n = inp["posi"].shape[0]
    coarse = torch.rand(n // 64 + 1, generator=g, device=GPU)
    r = coarse.repeat_interleave(64)[:n] * 0.8 + 0.2 * torch.rand(n, generator=g, device=GPU)
    r[inp["tag"] != 1] = 2.0
    k = max(1, int(case["fraction"] * int((inp["tag"] == 1).sum())))
    act = torch.zeros(n, dtype=torch.uint8, device=GPU)
    act[torch.argsort(r)[:k]] = 1
    return act


def uneven_inputs(case, seed):
    """Leaf cubes on distinct sites of a periodic lattice, occupancies
    log-uniform in 1..256, targets with 1..400 sources within 7 sites."""
    g = generator(seed)
    m = case["lattice"]
    cell = BOX / m
    pool = min(65536, m ** 3 // 2)
    sites = torch.argsort(torch.rand(m ** 3, generator=g, device=GPU))[:pool]
    ijk = torch.stack([sites // (m * m), sites // m % m, sites % m], 1)
    occ = (256.0 ** ((torch.arange(pool, device=GPU, dtype=torch.float64) + 0.5) / pool)).long().clamp(1, 256)
    occ = occ[torch.argsort(torch.rand(pool, generator=g, device=GPU))]
    owner = torch.repeat_interleave(torch.arange(pool, device=GPU), occ)
    pos = (ijk[owner] + torch.rand(owner.numel(), 3, generator=g, device=GPU, dtype=torch.float64)) * cell
    site_of = torch.full((m ** 3,), -1, dtype=torch.long, device=GPU)
    site_of[sites] = torch.arange(pool, device=GPU)
    o = torch.arange(-7, 8, device=GPU)
    off = torch.stack(torch.meshgrid(o, o, o, indexing="ij"), -1).reshape(1, -1, 3)
    nt = case["pairs"] // 180 + 20
    tgt = torch.randint(pool, (nt,), generator=g, device=GPU)
    want = torch.randint(1, 401, (nt,), generator=g, device=GPU)
    q = (ijk[tgt][:, None] + off) % m
    cand = site_of[(q[..., 0] * m + q[..., 1]) * m + q[..., 2]]
    key = torch.rand(cand.shape, generator=g, device=GPU) + 2.0 * (cand < 0)
    pick = torch.argsort(key, 1)[:, :400]
    src = torch.gather(cand, 1, pick)
    ok = (torch.arange(400, device=GPU)[None] < want[:, None]) & (src >= 0)
    t = tgt[:, None].expand_as(src)[ok][:case["pairs"]]
    s = src[ok][:case["pairs"]]
    return {"pos": pos, "ip": occ.cumsum(0) - occ, "np": occ, "t": t, "s": s, "rs": 1.25 * cell,
            "eps": cell / 40.0 if case["soft"] == "plummer" else 0.03 * cell}


def multipole_inputs(case, seed):
    """Cells of a tree with multipoles of the size that their particles give."""
    inp = tree_list(case, seed)
    tree = inp["tree"]
    g = generator(seed + 104729)
    w = tree["width"].double()
    n = torch.cat([tree["np"].double(), torch.full((tree["sons"].shape[0],), 2.0 * case["maxleaf"], device=GPU, dtype=torch.float64)])
    size = w.prod(1) ** (1 / 3)
    order = torch.tensor([0] + [1] * 3 + [2] * 6 + [3] * 10, device=GPU)
    scale = torch.tensor([1.0, 0.1, 0.04, 0.01], device=GPU, dtype=torch.float64)[order] * size[:, None] ** order
    z = torch.randn(w.shape[0], 20, generator=g, device=GPU, dtype=torch.float64)
    z[:, 0] = 1.0
    z[:, [4, 7, 9]] = 1.0 + 0.3 * z[:, [4, 7, 9]]     # the diagonal second moments are positive
    inp["M"] = (MASS * n[:, None] * scale * z).float()
    return inp


def law_of(case, eps, rs, box=0.0):
    return pp.ForceLaw(eps=eps, rs=rs, mass=MASS, box=box,
                       softening=pp.SOFT_PLUMMER if case.get("soft") == "plummer" else pp.SOFT_REF,
                       law={"table": pp.LAW_TABLE, "linear": pp.LAW_LINEAR}[case.get("law", "table")])


def host(x, dtype=np.int32):
    return x.cpu().numpy().astype(dtype, copy=False)


# ----------------------------------------------------------- prepare and run

def prepare(case, seed):
    """The context a program keeps, and what it holds on the host before the call."""
    ctx = pp.Context(0)
    st = {"ctx": ctx, "kind": case["kind"]}
    if case["kind"] == "uneven":
        u = uneven_inputs(case, seed)
        ctx.set_law(law_of(case, u["eps"], u["rs"], BOX))
        ctx.set_particles(host(u["pos"], np.float64), host(u["ip"]), host(u["np"]))
        ctx.set_tasks(host(u["t"]), host(u["s"]))
        ctx.prepare()
        st["kind"] = "force"
        return st
    rs, cutoff, step, eps = scales(case)
    ctx.set_law(law_of(case, eps, rs))
    st.update(step=step, rs=rs)
    if case["kind"] in ("step", "tree", "mesh"):
        posi, tag = particles(case, seed)
        lo, hi = bounds(posi, step)
        st.update(posi=host(posi), tag=host(tag), lo=lo, hi=hi, cutoff=cutoff)
        if case["kind"] == "mesh":
            if not case["tags"]:                     # a program without ghosts passes its local particles only
                st["posi"], st["tag"] = st["posi"][st["tag"] == 1], None
            st["mesh"] = case["mesh"]
        else:
            st.update(maxleaf=case["maxleaf"], theta=case["theta"], mesh=case["n1"] + case["n1"] % 2)
        if case["kind"] == "tree":                   # the arrays of a program in C, sized once for its lists
            n = posi.shape[0]
            cells = 64 + 4 * n // case["maxleaf"]
            pairs = 4096 + int(6000.0 * n / case["maxleaf"] ** 1.5)
            ints = {"perm": n, "leaf_ip": cells, "leaf_np": cells, "leaf_active": cells, "node_son": 2 * cells, "task_t": pairs, "task_s": pairs}
            st["out"] = {k: np.zeros(v, np.int32) for k, v in ints.items()}
            st["out"].update({k: np.zeros(3 * cells, np.float32) for k in ("leaf_center", "leaf_width", "node_center", "node_width")})
            st.update(cells=cells, pairs=pairs)
        return st
    if case["kind"] == "multipole":
        inp = multipole_inputs(case, seed)
        nl = inp["ip"].numel()
        center = host(inp["tree"]["center"], np.float32)
        st.update(center=center, leaf_center=np.ascontiguousarray(center[:nl]), M=host(inp["M"], np.float32),
                  t=host(inp["mt"]), s=host(inp["ms"]), nleaf=nl)
        ctx.set_particles(host(inp["posi"].double() * step, np.float64), host(inp["ip"]), host(inp["np"]))
        return st
    inp = tree_list(case, seed)
    if case["kind"] == "hostlists":
        body = np.zeros(inp["posi"].shape[0], dtype=[("posi", np.int32, 3), ("rest", np.int32, 7)])
        body["posi"] = host(inp["posi"])
        st.update(body=body, ip=host(inp["ip"]), num=host(inp["np"]), t=host(inp["t"]), s=host(inp["s"]))
        return st
    ctx.set_particles(host(inp["posi"].double() * step, np.float64), host(inp["ip"]), host(inp["np"]))
    ctx.set_tasks(host(inp["t"]), host(inp["s"]))
    if case["kind"] == "active":
        st["act"] = host(active_levels(case, seed, inp), np.uint8)
    ctx.prepare()
    return st


def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "force":
        ctx.zero_acc()
        ctx.compute()
        return ctx.acc_f32_soa()
    if kind == "active":
        ctx.set_active(st["act"], 1)
        ctx.zero_acc()
        ctx.compute()
        return ctx.acc_f32_soa()
    if kind == "hostlists":
        ctx.set_particles_i32(st["body"], st["step"], st["ip"], st["num"])
        ctx.set_tasks(st["t"], st["s"])
        ctx.compute()
        return ctx.acc_f32_soa()
    if kind == "multipole":
        L, _ = ctx.m2l(st["center"], st["M"], st["t"], st["s"], st["rs"])
        ctx.zero_acc()
        ctx.l2p(L[:st["nleaf"]], st["leaf_center"])
        return L, ctx.acc()
    if kind == "mesh":
        return ctx.pm_forces(st["posi"], st["tag"], st["step"], BOX, st["mesh"], st["rs"], MASS)[0]
    nleaf, nnode = ctx.build_tree(st["posi"], st["tag"], st["step"], st["maxleaf"], st["lo"], st["hi"])
    ntask = ctx.walk_tree(st["theta"], st["cutoff"])
    if kind == "tree":
        if max(nleaf, nnode) > st["cells"] or ntask > st["pairs"]:
            raise ValueError("the program's arrays are too small")
        o, lib = st["out"], pp.load()
        at = [o[k].ctypes.data for k in ("perm", "leaf_ip", "leaf_np", "leaf_active", "leaf_center", "leaf_width", "node_son",
                                         "node_center", "node_width")]
        if lib.pp2p_get_tree(ctx._h, *at) or lib.pp2p_get_tasks(ctx._h, None, o["task_t"].ctypes.data, o["task_s"].ctypes.data):
            raise RuntimeError(lib.pp2p_last_error().decode())
        return nleaf, nnode, ntask, o
    ctx.compute()
    ctx.fmm_short()
    ctx.pm_add_tree(BOX, st["mesh"], st["rs"], MASS)
    return ctx.get_tree()["perm"], ctx.acc_f32_soa()


# -------------------------------------------------------------------- figures

def counts(case):
    """Particles with ghosts, pairs inside the cutoff and leaf pairs, about."""
    if case["kind"] == "uneven":
        return case["lattice"] ** 3 * 12, case["pairs"] * 46.0 ** 2 * 0.5, case["pairs"]
    n1 = case["n1"]
    n = n1 ** 3 * (1.0 + 2 * 4.5 * 1.25 / n1) ** 3
    crowd = 3.6 if case["dist"] == "clustered" else 1.0
    near = n1 ** 3 * 4.19 * (2 * UCUT * 1.25) ** 3 * crowd
    leaf = 0.72 * case.get("maxleaf", 32)
    return n, near, 1.8 * near / (leaf * leaf)


def n1cube(case):
    return float(case["n1"] ** 3)


def work(case):
    """Bytes: inputs read and outputs written once (intermediate lists not
    counted); operations: 48 per pair inside the cutoff, 5 N log2 N per
    transform, about 700 per M2L translation."""
    n, near, tasks = counts(case)
    kind = case["kind"]
    if kind == "tree":
        return {"bytes": 20.0 * n + 8.0 * tasks, "flops": 3.0 * n * math.log2(max(2.0, n / case["maxleaf"]))}
    if kind == "multipole":
        n, cells = n1cube(case), 2.0 * n1cube(case) / (0.72 * case["maxleaf"])
        return {"bytes": 172.0 * cells + 48.0 * n, "flops": 700.0 * 20 * cells + 60.0 * n}
    m = case.get("mesh", case.get("n1", 0))
    mesh = {"bytes": 28.0 * n, "flops": 10.0 * m ** 3 * math.log2(max(2, m)) * 3 + 200.0 * n}
    if kind == "mesh":
        return mesh
    if kind == "step":
        return {"bytes": 32.0 * n, "flops": 48.0 * near + mesh["flops"]}
    if kind == "active":
        return {"bytes": 29.0 * n + 8.0 * tasks * case["fraction"], "flops": 48.0 * near * case["fraction"]}
    return {"bytes": 28.0 * n + 8.0 * tasks, "flops": 48.0 * near}


# ---------------------------------------------------------------------- exact

def pair_forces(pos, ip, num, t, s, eps, rs, plummer_soft, box=0.0):
    """The short-range pair sums over the listed leaf pairs in FP64."""
    n, nl = pos.shape[0], ip.numel()
    acc = torch.zeros(n + 1, 3, dtype=torch.float64, device=GPU)
    pad = torch.cat([pos, torch.full((1, 3), 1e6, dtype=torch.float64, device=GPU)])
    ok = (num[t] > 0) & (num[s] > 0)
    t, s = t[ok], s[ok]
    by = torch.argsort(num[t] // 8 * 4096 + num[s] // 8, stable=True)
    t, s = t[by], s[by]
    if not t.numel():
        return acc[:n]
    nt, ns = (num[t] // 8 * 8 + 7).cpu().numpy(), (num[s] // 8 * 8 + 7).cpu().numpy()
    rc2 = (2 * rs * UCUT) ** 2
    k = 0
    while k < t.numel():
        e = min(t.numel(), k + max(1, (1 << 26) // int(nt[k] * ns[k])))
        same = np.flatnonzero((nt[k:e] != nt[k]) | (ns[k:e] != ns[k]))
        e = k + int(same[0]) if same.size else e
        a, b = torch.arange(int(nt[k]), device=GPU), torch.arange(int(ns[k]), device=GPU)
        i = torch.where(a[None] < num[t[k:e]][:, None], ip[t[k:e]][:, None] + a[None], n)
        j = torch.where(b[None] < num[s[k:e]][:, None], ip[s[k:e]][:, None] + b[None], n)
        d = [pad[j, c][:, None, :] - pad[i, c][:, :, None] for c in range(3)]
        if box:
            d = [x - box * torch.round(x / box) for x in d]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        r2 = r2 + eps * eps if plummer_soft else r2.clamp_min(eps * eps)
        r = r2.sqrt()
        u = r / (2 * rs)
        f = (torch.special.erfc(u) + (2 / math.sqrt(math.pi)) * u * torch.exp(-u * u)) / (r2 * r)
        f = torch.where((r2 < rc2) & (i < n)[:, :, None] & (j < n)[:, None, :], f, 0.0)
        acc.index_add_(0, i.reshape(-1), torch.stack([(f * x).sum(2) for x in d], -1).reshape(-1, 3))
        k = e
    return MASS * acc[:n]


# exponents of the 20 coefficients, orders 0 to 3, z last
EXPS = [(a, b, n - a - b) for n in range(4) for a in range(n, -1, -1) for b in range(n - a, -1, -1)]


def exact_multipole(case, seed):
    inp = multipole_inputs(case, seed)
    rs, _, step, _ = scales(case)
    nl = inp["ip"].numel()
    c, M = inp["tree"]["center"].double(), inp["M"].double()
    rs = float(np.float32(rs))
    L = torch.zeros_like(M)
    at = {e: k for k, e in enumerate(EXPS)}
    for k in range(0, inp["mt"].numel(), 1 << 20):
        t, s = inp["mt"][k:k + (1 << 20)], inp["ms"][k:k + (1 << 20)]
        x = c[t] - c[s]
        keep = x.square().sum(1) >= 1.0              # closer cells add nothing, as in the reference
        t, s, x = t[keep], s[keep], x[keep]
        r = x.norm(dim=1)
        # f_k = ((1/r) d/dr)^k of erfc(r / 2 rs) / r
        E, q = torch.special.erfc(r / (2 * rs)), torch.exp(-r * r / (4 * rs * rs)) / (rs * math.sqrt(math.pi))
        h = 1 / (2 * rs * rs)
        f = [E / r, -E / r ** 3 - q / r ** 2, 3 * E / r ** 5 + 3 * q / r ** 4 + q * h / r ** 2,
             -15 * E / r ** 7 - 15 * q / r ** 6 - 5 * q * h / r ** 4 - q * h * h / r ** 2]
        D = []
        for e in EXPS:
            ax = [d for d in range(3) for _ in range(e[d])]
            y = [x[:, d] for d in ax]
            if len(ax) < 2:
                D.append(f[len(ax)] * (y[0] if y else 1.0))
            elif len(ax) == 2:
                D.append(f[2] * y[0] * y[1] + (f[1] if ax[0] == ax[1] else 0.0))
            else:
                v = f[3] * y[0] * y[1] * y[2]
                for i, j, k2 in ((0, 1, 2), (0, 2, 1), (1, 2, 0)):
                    if ax[i] == ax[j]:
                        v = v + f[2] * y[k2]
                D.append(v)
        m = M[s]
        out = torch.zeros(t.numel(), 20, dtype=torch.float64, device=GPU)
        for b, eb in enumerate(EXPS):
            for a, ea in enumerate(EXPS):
                if sum(ea) + sum(eb) <= 3:
                    out[:, b] += m[:, a] * D[at[tuple(p + q2 for p, q2 in zip(ea, eb))]]
        L.index_add_(0, t, out)
    leaf = torch.repeat_interleave(torch.arange(nl, device=GPU), inp["np"])
    d = inp["posi"].double() * step - c[leaf]
    F = torch.zeros_like(d)
    for i in range(3):
        for e in EXPS:
            if sum(e) <= 2:
                up = tuple(v + (k == i) for k, v in enumerate(e))
                F[:, i] += L[leaf, at[up]] * (d ** torch.tensor(e, device=GPU)).prod(1) / math.prod(math.factorial(v) for v in e)
    return L, F


def exact_mesh(case, seed):
    posi, tag = particles(case, seed)
    rs, _, step, _ = scales(case)
    local = tag == 1
    N, box, pi = case["mesh"], BOX, float(np.float32(3.1415926))
    x = (posi[local].double() * step).float().double() * (N / box)          # the entry takes FP32 positions
    own = torch.floor(x).long()
    w = x - own - 0.5
    side = torch.where(w > 0, own + 1, own - 1)
    cells, wts = (own % N, side % N), (1 - w.abs(), w.abs())
    m = float(np.float32(MASS))
    corners = [(((cells[i][:, 0] * N + cells[j][:, 1]) * N + cells[k][:, 2]), wts[i][:, 0] * wts[j][:, 1] * wts[k][:, 2])
               for i in (0, 1) for j in (0, 1) for k in (0, 1)]
    rho = torch.zeros(N ** 3, dtype=torch.float64, device=GPU)
    for cell, wt in corners:
        rho.index_add_(0, cell, m * wt)
    k = torch.arange(N, device=GPU, dtype=torch.float64)
    k = torch.where(k > N // 2, k - N, k)
    ks = (k[:, None, None], k[None, :, None], k[None, None, :N // 2 + 1].abs())
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    sinc = 1.0
    for q in ks:
        sinc = sinc * torch.where(q == 0, 1.0, torch.sin(pi * q / N) / torch.where(q == 0, 1.0, pi * q / N))
    G = torch.exp(-k2 * (2 * pi * float(np.float32(rs)) / box) ** 2) / torch.where(k2 == 0, 1.0, k2) / sinc ** 4 * (box * box / pi) * (1 / box) ** 3
    G[0, 0, 0] = 0.0
    pot = torch.fft.irfftn(torch.fft.rfftn(rho.reshape(N, N, N)) * G, s=(N, N, N)) * float(N) ** 3
    h = 0.5 * N / box
    acc = torch.zeros(posi.shape[0], 3, dtype=torch.float64, device=GPU)
    for d in range(3):
        g = (4 / 3) * h * (pot.roll(-1, d) - pot.roll(1, d)) - (1 / 6) * h * (pot.roll(-2, d) - pot.roll(2, d))
        acc[local, d] = sum(wt * g.reshape(-1)[cell] for cell, wt in corners)
    return acc if case["tags"] else acc[local]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "tree"):                     # whole calls: their parts are the other cases; trees and lists are whole numbers
        return None
    if kind == "multipole":
        return exact_multipole(case, seed)
    if kind == "mesh":
        return exact_mesh(case, seed)
    soft = case["soft"] == "plummer"
    if kind == "uneven":
        u = uneven_inputs(case, seed)
        return pair_forces(u["pos"], u["ip"], u["np"], u["t"], u["s"], u["eps"], u["rs"], soft, BOX).T.contiguous()
    inp = tree_list(case, seed)
    rs, _, step, eps = scales(case)
    t, s = inp["t"], inp["s"]
    if kind == "active":
        act = active_levels(case, seed, inp) == 1
        c = torch.cat([torch.zeros(1, dtype=torch.long, device=GPU), act.long().cumsum(0)])
        has = c[inp["ip"] + inp["np"]] > c[inp["ip"]]
        t, s = t[has[t]], s[has[t]]
    acc = pair_forces(inp["posi"].double() * step, inp["ip"], inp["np"], t, s, eps, rs, soft)
    if kind == "active":
        acc[~act] = 0.0
    return acc.T.contiguous()
