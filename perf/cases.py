"""The work a user of this library has it do, as cases that can be timed.

A case is a dict of plain values; its "kind" names the entry points it takes:

  one      hbt_unbind_one: one subhalo from host buffers (Subhalo_t::Unbind)
  batch    hbt_unbind_batch: a rank's subhalos resident on the device
  share    hbt_id_to_index and hbt_unbind_batch_indexed: source-ID lists into a
           shuffled snapshot (RefineParticles of one rank's share)
  nested   hbt_unbind_batch: a host with satellites nested in it
  tree     hbt_tree_potential: a halo's potential at its own particles
  pairs    hbt_direct_potential: exact pair sums, the precision study
  props    hbt_subhalo_properties: profiles and shapes of bound lists
  mask     hbt_mask_subhalos: exclusive ownership of overlapping lists
  merge    hbt_merge_subhalos: trapped subhalos merged, their hosts unbound again

Inputs follow the workloads of hbtplus_amd/synth.py (NFW haloes with Jeans
velocities, contaminants, periodic 100 Mpc/h box), generated on the GPU.  The
sizes of a population are the quantiles of its size law, so every seed has the
same sizes and other particles.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from hbtplus_amd import abi, synth
from hbtplus_amd.device import GpuUnbinder

DEV = "cuda:0"
BOX = 1.0e5
MASS = synth.PARTICLE_MASS
G = float(np.float32(synth.G_DEFAULT))  # as the parameter record holds it


def listed():
    return [
        # one small subhalo through the per-subhalo interface: the reference's
        # Unbind call on the sizes most subhalos have, all launches and waits
        dict(name="one_300", kind="one", n=300),
        # the same on the single 24,000-particle halo (20,000 NFW + 20%)
        dict(name="one_24k", kind="one", n=20_000),
        # a mid-size rank: 5,000 subhalos of the power law, 1.5 M particles
        dict(name="batch_5k", kind="batch", n=5_000, law="power", precision="fast"),
        # many small groups, log-uniform on [20, 4096] with Gaussian contaminants
        dict(name="batch_50k_small", kind="batch", n=50_000, law="small", precision="fast"),
        # one rank's full share: 200,000 subhalos by ID out of a 70 M snapshot
        dict(name="share_200k", kind="share", n=200_000, sample=0),
        # the reference's default mode, potentials from 1000 sampled particles
        dict(name="share_20k_sampled", kind="share", n=20_000, sample=1000),
        # a cluster: 4 M particles and 200 satellites unbound before it
        dict(name="nested_4M", kind="nested", n=4_000_000, nsat=200),
        # the potential of one large halo at its particles, periodic box
        dict(name="tree_100k", kind="tree", n=100_000, periodic=True),
        # the precision study's three pair sums over 600 small subhalos
        dict(name="pairs_600", kind="pairs", n=600),
        # profiles and shapes after the unbinding of 20,000 subhalos
        dict(name="props_20k", kind="props", n=20_000),
        # 1,000 host groups whose lists overlap, 4 M entries
        dict(name="mask_1000", kind="mask", n=1_000),
        # 300 host groups after their unbinding, half the subhalos trapped
        dict(name="merge_300", kind="merge", n=300),
    ]


def _log(rng, lo, hi):
    """A size spread evenly over its logarithm, odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["one", "batch", "batch", "share", "share", "nested", "tree", "pairs", "props", "mask", "merge"])
    if kind == "one":
        return dict(kind=kind, n=_log(rng, 20, 200_000))
    if kind == "batch":
        law = rng.choice(["power", "small"])
        precision = rng.choice(["fast", "fast", "fast", "replay"])
        # bit-level certification runs on catalogues of test size
        return dict(kind=kind, n=_log(rng, 50, 2_000 if precision == "replay" else 50_000), law=law, precision=precision)
    if kind == "share":
        return dict(kind=kind, n=_log(rng, 500, 100_000), sample=rng.choice([0, 0, 1000]))
    if kind == "nested":
        return dict(kind=kind, n=_log(rng, 50_000, 4_000_000), nsat=rng.randint(5, 200))
    if kind == "tree":
        return dict(kind=kind, n=_log(rng, 200, 400_000), periodic=rng.choice([False, True]))
    if kind == "pairs":
        return dict(kind=kind, n=_log(rng, 20, 3_000))
    if kind == "props":
        return dict(kind=kind, n=_log(rng, 100, 100_000))
    if kind == "mask":
        return dict(kind=kind, n=_log(rng, 20, 2_000))
    return dict(kind=kind, n=_log(rng, 10, 500))


# ---- inputs -------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(g, n):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _unit(g, n):
    v = _normal(g, n, 3)
    return v / v.norm(dim=1, keepdim=True)


def _mu(x):
    return torch.log1p(x) - x / (1.0 + x)


def _counts(n, law):
    """Sizes of n subhalos: the quantiles of the size law."""
    u = (np.arange(n) + 0.5) / n
    if law == "power":  # dN/dN_p ~ N_p^-1.9 on [20, 2e5]
        a, b = 20.0 ** -0.9, 2.0e5 ** -0.9
        return np.rint((a + u * (b - a)) ** (-1.0 / 0.9)).astype(np.int64)
    return np.rint(np.exp(np.log(20.0) + u * np.log(4096.0 / 20.0))).astype(np.int64)


def _nfw(g, owner, counts, conc, r200):
    """Relative positions and velocities of NFW members, one row per owner
    entry: radii by bisection of the enclosed mass, isotropic Jeans dispersions."""
    c = conc[owner]
    target = _rand(g, len(owner)) * _mu(c)
    lo = torch.full_like(c, -14.0)
    hi = torch.zeros_like(c)
    for _ in range(30):
        mid = 0.5 * (lo + hi)
        below = _mu(c * mid.exp()) < target
        lo = torch.where(below, mid, lo)
        hi = torch.where(below, hi, mid)
    y = 0.5 * (lo + hi)  # ln(x / c)
    x = c * y.exp()
    rs = r200[owner] / c
    jeans = synth._JeansTable(float(conc.min()), float(conc.max()))
    tab = torch.from_numpy(jeans.tab).to(DEV)
    kc = ((c.log() - jeans.lc[0]) / (jeans.lc[1] - jeans.lc[0])).round().long().clamp(0, len(jeans.lc) - 1)
    fy = (y.clamp(min=math.log(1e-6)) - jeans.ly[0]) / (jeans.ly[1] - jeans.ly[0])
    jy = fy.floor().long().clamp(0, len(jeans.ly) - 2)
    w = fy - jy
    s2 = tab[kc, jy] * (1 - w) + tab[kc, jy + 1] * w
    v2 = G * MASS * counts[owner].double() / (rs * _mu(c))
    pos = _unit(g, len(owner)) * (x * rs)[:, None]
    vel = _normal(g, len(owner), 3) * (v2 * s2).clamp(min=0).sqrt()[:, None]
    return pos, vel, x, v2


def _population(g, counts_np, law):
    """A population of subhalos with contaminants, grouped by subhalo and in
    random order inside each: (owner, total counts, positions, velocities,
    centres, bulk velocities).  Power law: log-normal concentrations, 20%
    contaminants at three times the escape speed; small groups: c = 10, 15%
    contaminants at 1000 km/s with a 300 km/s offset."""
    n = len(counts_np)
    counts = torch.from_numpy(counts_np).to(DEV)
    power = law == "power"
    conc = 10.0 * torch.exp(0.3 * _normal(g, n)) if power else torch.full((n,), 10.0, device=DEV, dtype=torch.float64)
    r200 = 200.0 * (counts.double() / 2.0e4) ** (1.0 / 3.0)
    owner = torch.repeat_interleave(torch.arange(n, device=DEV), counts)
    rp, rv, _, _ = _nfw(g, owner, counts, conc, r200)
    ncont = torch.from_numpy(np.rint((0.2 if power else 0.15) * counts_np).astype(np.int64)).to(DEV)
    co = torch.repeat_interleave(torch.arange(n, device=DEV), ncont)
    cp = _unit(g, len(co)) * (r200[co] * _rand(g, len(co)) ** (1.0 / 3.0))[:, None]
    if power:
        c, rs = conc[co], r200[co] / conc[co]
        x = (cp.norm(dim=1) / rs).clamp(min=1e-9)
        v2 = G * MASS * counts[co].double() / (rs * _mu(c))
        vesc = (2.0 * v2 * (torch.log1p(x) / x - 1.0 / (1.0 + c)).clamp(min=0)).sqrt()
        cv = _unit(g, len(co)) * (3.0 * vesc)[:, None]
    else:
        cv = _normal(g, len(co), 3) * 1000.0
        cv[:, 0] += 300.0
    own = torch.cat([owner, co])
    order = torch.argsort(own + _rand(g, len(own)))
    centres = _rand(g, 3 * n).view(n, 3) * BOX
    bulk = _normal(g, n, 3) * 300.0
    return (own[order], counts_np + np.rint((0.2 if power else 0.15) * counts_np).astype(np.int64),
            torch.cat([rp, cp])[order], torch.cat([rv, cv])[order], centres, bulk)


def _ids(g, n):
    """n distinct particle IDs, scattered over [0, 2^62)."""
    perm = torch.randperm(n, generator=g, device=DEV)
    return (perm * 2654435761 + 1000003) & ((1 << 62) - 1)


def _columns(pos, vel, ids):
    f = lambda v: v.to(torch.float32).contiguous()  # noqa: E731
    n = len(pos)
    return dict(id=ids, x=f(pos[:, 0]), y=f(pos[:, 1]), z=f(pos[:, 2]), vx=f(vel[:, 0]), vy=f(vel[:, 1]),
                vz=f(vel[:, 2]), mass=torch.full((n,), MASS, device=DEV, dtype=torch.float32),
                type=torch.ones(n, device=DEV, dtype=torch.int32))


def _records(counts, centres, bulk, parent=None):
    """Subhalo records whose frame is the previous snapshot's: centre and bulk velocity."""
    n = len(counts)
    subs = np.zeros(n, abi.SUB_DTYPE)
    subs["offset"] = np.concatenate([[0], np.cumsum(counts)[:-1]])
    subs["count"] = counts
    subs["parent"] = -1 if parent is None else parent
    subs["nbound_prev"] = counts
    for f in ("sink_track_id", "snapshot_index_of_death", "snapshot_index_of_sink"):
        subs[f] = -1
    subs["ref_pos"] = subs["mostbound_pos"] = centres.to(torch.float32).cpu().numpy()
    subs["ref_vel"] = subs["mostbound_vel"] = bulk.to(torch.float32).cpu().numpy()
    return subs


def _handle(cols, subs, **more):
    """What GpuUnbinder.upload returns, for columns that are on the device already."""
    total = abi.plan_batch(subs)
    return dict(cols=cols, subs_host=subs, total=total, subs0=torch.from_numpy(subs.view(np.uint8)).to(DEV),
                ps=abi.particles_struct(cols, ptr=lambda t: t.data_ptr()), **more)


def _params(**kw):
    return abi.make_params(**{**dict(softening=0.5, open_angle=0.45, periodic=1, box_size=BOX), **kw})


def _prepare_one(case, g):
    own, counts, rp, rv, _, _ = _population(g, np.array([case["n"]]), "power")
    cols = {k: v.cpu().numpy() for k, v in _columns(rp, rv, _ids(g, len(own))).items()}
    zero = torch.zeros(1, 3, device=DEV, dtype=torch.float64)
    return dict(U=GpuUnbinder(_params(periodic=0)), cols=cols, sub=_records(counts, zero, zero))


def _prepare_batch(case, g):
    own, counts, rp, rv, cen, bulk = _population(g, _counts(case["n"], case["law"]), case["law"])
    cols = _columns((cen[own] + rp) % BOX, bulk[own] + rv, _ids(g, len(own)))
    precision = abi.HBT_PREC_REPLAY if case["precision"] == "replay" else abi.HBT_PREC_FAST
    return dict(U=GpuUnbinder(_params(precision=precision)), h=_handle(cols, _records(counts, cen, bulk)))


def _prepare_share(case, g):
    own, counts, rp, rv, cen, bulk = _population(g, _counts(case["n"], "power"), "power")
    nlist, nbg = len(own), len(own) // 10  # a tenth of the listed particles as background
    perm = torch.randperm(nlist + nbg, generator=g, device=DEV)
    pos = torch.cat([(cen[own] + rp) % BOX, _rand(g, 3 * nbg).view(nbg, 3) * BOX])
    vel = torch.cat([bulk[own] + rv, _normal(g, nbg, 3) * 300.0])
    ids = _ids(g, nlist + nbg)
    cols = _columns(pos[perm], vel[perm], ids[perm])
    h = _handle(cols, _records(counts, cen, bulk), ids=ids[:nlist].clone())
    return dict(U=GpuUnbinder(_params(max_sample_size=case["sample"])), h=h, sample=case["sample"])


def _prepare_nested(case, g):
    n, nsat = case["n"], case["nsat"]
    u = (np.arange(nsat) + 0.5) / nsat
    lo, hi = max(50.0, n / 4000.0), max(500.0, n / 40.0)  # satellites of a 4M host: 1e3 .. 1e5
    sizes = np.rint((lo ** -0.9 + u * (hi ** -0.9 - lo ** -0.9)) ** (-1.0 / 0.9)).astype(np.int64)
    counts_np = np.concatenate([[n], sizes])
    counts = torch.from_numpy(counts_np).to(DEV)
    conc = torch.full((nsat + 1,), 10.0, device=DEV, dtype=torch.float64)
    conc[0] = 5.0
    r200 = 200.0 * (counts.double() / 2.0e4) ** (1.0 / 3.0)
    own = torch.repeat_interleave(torch.arange(nsat + 1, device=DEV), counts)
    rp, rv, _, v2 = _nfw(g, own, counts, conc, r200)
    cen = _unit(g, nsat + 1) * (r200[0] * _rand(g, nsat + 1) ** (1.0 / 3.0))[:, None]
    bulk = _normal(g, nsat + 1, 3) * (0.6 * v2[0].sqrt())
    cen[0] = 0.0
    bulk[0] = 0.0
    cols = _columns(cen[own] + rp, bulk[own] + rv, _ids(g, len(own)))
    parent = np.concatenate([[-1], np.zeros(nsat, np.int64)])
    return dict(U=GpuUnbinder(_params(softening=1.0, periodic=0)), h=_handle(cols, _records(counts_np, cen, bulk, parent)))


def _halo_columns(case, g):
    own, _, rp, rv, cen, _ = _population(g, np.array([case["n"]]), "power")
    return _columns((cen[own] + rp) % BOX if case.get("periodic", True) else rp, rv, _ids(g, len(own)))


def _prepare_tree(case, g):
    cols = _halo_columns(case, g)
    return dict(U=GpuUnbinder(_params(periodic=int(case["periodic"]))), cols=cols)


def _pairs_inputs(case, g):
    own, counts, rp, rv, cen, bulk = _population(g, _counts(case["n"], "small"), "small")
    return counts, _columns((cen[own] + rp) % BOX, bulk[own] + rv, _ids(g, len(own)))


def _prepare_pairs(case, g):
    counts, cols = _pairs_inputs(case, g)
    seg = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)])).to(DEV)
    return dict(U=GpuUnbinder(_params()), cols=cols, seg=seg)


def _props_inputs(case, g):
    """Bound lists as the unbinding leaves them: NFW members with negative
    energy in their halo's potential, most bound first, in a shuffled snapshot."""
    counts_np = _counts(case["n"], "power")
    n = len(counts_np)
    counts = torch.from_numpy(counts_np).to(DEV)
    conc = 10.0 * torch.exp(0.3 * _normal(g, n))
    r200 = 200.0 * (counts.double() / 2.0e4) ** (1.0 / 3.0)
    own = torch.repeat_interleave(torch.arange(n, device=DEV), counts)
    rp, rv, x, v2 = _nfw(g, own, counts, conc, r200)
    energy = 0.5 * (rv * rv).sum(1) / v2 - torch.log1p(x) / x + 1.0 / (1.0 + conc[own])
    cen = _rand(g, 3 * n).view(n, 3) * BOX
    bulk = _normal(g, n, 3) * 300.0
    perm = torch.randperm(len(own), generator=g, device=DEV)  # list entry -> snapshot position
    place = torch.empty_like(perm)
    place[perm] = torch.arange(len(perm), device=DEV)
    cols = _columns(((cen[own] + rp) % BOX)[perm], (bulk[own] + rv)[perm], _ids(g, len(own)))
    # scaled into (0, 1): bound particles of a subhalo sort before its unbound ones
    order = torch.argsort(own + 0.5 + 0.499 * torch.tanh(0.2 * energy))
    nbound = torch.zeros(n, device=DEV, dtype=torch.int64).index_add_(0, own, (energy < 0).long()).cpu().numpy()
    out_index = place[order]
    subs = _records(counts_np, cen, bulk)
    subs["out_offset"] = subs["offset"]
    subs["nbound"] = nbound
    subs["mbound"] = (nbound * np.float64(np.float32(MASS))).astype(np.float32)
    first = out_index[torch.from_numpy(subs["offset"].copy()).to(DEV)]
    subs["mostbound_pos"] = torch.stack([cols[k][first] for k in "xyz"], 1).cpu().numpy()
    return cols, subs, out_index


PROPS_HZ = float(np.float32(0.1))  # km/s per kpc/h, today's expansion rate


def _prepare_props(case, g):
    cols, subs, out_index = _props_inputs(case, g)
    h = dict(cols=cols, subs_host=subs, ps=abi.particles_struct(cols, ptr=lambda t: t.data_ptr()))
    return dict(U=GpuUnbinder(_params(hz=PROPS_HZ)), h=h,
                out=(torch.from_numpy(subs.view(np.uint8)).to(DEV), out_index, None))


def _prepare_mask(case, g):
    """Host groups whose lists are drawn from one pool of IDs each, so that
    they overlap and repeat: 1 to 12 subhalos a group, nests inside it, some
    orphans (they claim nothing), some null IDs, a few field subhalos.  The
    structure is the same for every seed, the drawn IDs are not."""
    rng = np.random.Generator(np.random.Philox(key=case["n"]))
    pool = 4000
    count, parent, nprev, grp = [], [], [], []
    for k in range(case["n"]):
        ns, first = int(rng.integers(1, 13)), len(count)
        for i in range(ns):
            n = int(rng.integers(0, 2 * max(2, pool // ns)))
            head = i == 0 or rng.random() < 0.3
            parent.append(-1 if head else first + int(rng.integers(0, i)))
            nprev.append(1 if rng.random() < 0.15 else max(2, n))
            count.append(n)
            grp.append(k)
    for i in range(5):
        count, parent, nprev, grp = count + [50], parent + [-1], nprev + [50], grp + [-1]
    count, grp = np.array(count, np.int64), np.array(grp, np.int64)
    zero = torch.zeros(len(count), 3, device=DEV, dtype=torch.float64)
    subs = _records(count, zero, zero, np.array(parent, np.int64))
    subs["nbound_prev"] = nprev
    group = torch.repeat_interleave(torch.from_numpy(grp).to(DEV), torch.from_numpy(count).to(DEV))
    n = len(group)
    ids = 1 + group.clamp(min=0) * pool + (_rand(g, n) * pool).long()
    ids[_rand(g, n) < 0.004] = -1
    pos = torch.zeros(n, 3, device=DEV)
    cols = _columns(pos, pos, ids)
    return dict(U=GpuUnbinder(_params()), cols=cols, ps=abi.particles_struct(cols, ptr=lambda t: t.data_ptr()),
                subs=subs, grp=grp)


# A host group of the merging case: (list size / 3, parent in the group,
# distance from the parent's centre and speed relative to it, in units of the
# central's r200 and v200); negative parent: a head.
_GROUP = [
    (1500, -1, 0.0, 0.0),     # the central
    (220, 0, 0.004, 0.005),   # a satellite at its core, with one at its own
    (60, 1, 0.002, 0.003),
    (400, 0, 0.5, 1.0),       # a satellite far out, with one at its core
    (65, 3, 0.002, 0.002),    # and one far from it
    (65, 3, 0.5, 1.0),
    (40, 0, 0.06, 0.0),       # too hot to stay bound
    (150, -1, 0.004, 0.005),  # a second head at the central's core, and one far out
    (100, -1, 0.8, 2.0),
]


def _prepare_merge(case, g):
    ng, per = case["n"], len(_GROUP)
    size = np.array([r[0] for r in _GROUP])
    # sizes vary by a quarter either way over the groups
    scale = 3.0 * (0.75 + 0.5 * (np.arange(ng) + 0.5) / ng)
    counts_np = np.rint(size[None, :] * scale[:, None]).astype(np.int64).reshape(-1)
    n = ng * per
    counts = torch.from_numpy(counts_np).to(DEV)
    r200 = 200.0 * (counts.double() / 2.0e4) ** (1.0 / 3.0)
    conc = torch.full((n,), 12.0, device=DEV, dtype=torch.float64)
    own = torch.repeat_interleave(torch.arange(n, device=DEV), counts)
    rp, rv, _, _ = _nfw(g, own, counts, conc, r200)
    rv = torch.where((own % per == 6)[:, None], 20.0 * rv, rv)
    cen = _rand(g, 3 * n).view(ng, per, 3) * BOX
    cen[::50, 0] = BOX - 2.0  # some groups lie across the box edge
    bulk = _normal(g, ng, per, 3) * 50.0
    r0 = r200.view(ng, per)[:, 0]
    v0 = (G * MASS * counts.double().view(ng, per)[:, 0] / r0).sqrt()
    for k, (_, p, dist, speed) in enumerate(_GROUP):
        if k:
            cen[:, k] = cen[:, max(p, 0)] + _unit(g, ng) * (dist * r0)[:, None]
            bulk[:, k] = bulk[:, max(p, 0)] + _unit(g, ng) * (speed * v0)[:, None]
    cen, bulk = cen.view(n, 3), bulk.view(n, 3)
    cols = _columns((cen[own] + rp) % BOX, bulk[own] + rv, _ids(g, len(own)))
    parent = np.array([r[1] for r in _GROUP])[None, :] + per * np.arange(ng)[:, None]
    parent = np.where(np.array([r[1] for r in _GROUP])[None, :] < 0, -1, parent).reshape(-1)
    U = GpuUnbinder(_params(snapshot_index=5))
    h = _handle(cols, _records(counts_np, cen % BOX, bulk, parent))
    rec, index, _ = U.unbind_device(h)
    subs = rec.cpu().numpy().view(abi.SUB_DTYPE).copy()
    # the lists after TruncateSource, end to end
    kept = subs["nsource"].astype(np.int64)
    offset = np.cumsum(kept) - kept
    at = np.repeat(subs["out_offset"] - offset, kept) + np.arange(kept.sum())
    subs["offset"], subs["count"] = offset, kept
    lists = index[torch.from_numpy(at).to(DEV)]
    return dict(U=U, hm=dict(cols=cols, ps=h["ps"], li=lists, n_list=len(at)), subs=subs, grp=np.repeat(np.arange(ng), per),
                out=torch.full((h["total"] + n,), -1, dtype=torch.int64, device=DEV))


def prepare(case, seed):
    kind = case["kind"]
    torch.cuda.set_device(0)
    make = dict(one=_prepare_one, batch=_prepare_batch, share=_prepare_share, nested=_prepare_nested, tree=_prepare_tree,
                pairs=_prepare_pairs, props=_prepare_props, mask=_prepare_mask, merge=_prepare_merge)[kind]
    return dict(make(case, _gen(seed)), kind=kind)


# ---- one pass -----------------------------------------------------------------

def _split(rec_i, rec_f):
    """The 60 words of each subhalo record (int32 and float32 views), whole numbers and floats apart."""
    return dict(ints=[rec_i[:, :12], rec_i[:, 24:42], rec_i[:, 54:]],
                frames=rec_f[:, 12:24], masses=rec_f[:, 42:49], energies=rec_f[:, 49:51], spin=rec_f[:, 51:54])


def _unbound(result):
    subs, index, energy = result
    return dict(_split(subs.view(torch.int32).view(-1, 60), subs.view(torch.float32).view(-1, 60)),
                index=index, energy=energy)


def _split_host(subs):
    return _split(subs.view(np.int32).reshape(-1, 60), subs.view(np.float32).reshape(-1, 60))


def run(state):
    kind, U = state["kind"], state["U"]
    if kind == "one":
        rec, index, energy = U.unbind_one(state["cols"], state["sub"])
        return dict(_split_host(rec), index=index, energy=energy)
    if kind in ("batch", "nested"):
        return _unbound(U.unbind_device(state["h"]))
    if kind == "share":
        if state["sample"]:
            U.set_rand_state(1, 0)  # each snapshot's shuffles from srand(1)
        return _unbound(U.unbind_indexed(state["h"], U.resolve_ids(state["h"])))
    if kind == "tree":
        c = state["cols"]
        n = len(c["x"])
        phi = torch.empty(n, dtype=torch.float64, device=DEV)
        p = [c[k].data_ptr() for k in ("x", "y", "z", "mass")]
        torch.cuda.synchronize()
        abi.check(U.lib.hbt_tree_potential(U.ctx, n, *p, n, *p, phi.data_ptr()), "hbt_tree_potential")
        return phi
    if kind == "pairs":
        c, seg = state["cols"], state["seg"]
        p = [c[k].data_ptr() for k in ("x", "y", "z", "mass")]
        out = []
        for mode in (abi.HBT_DIRECT_FP32, abi.HBT_DIRECT_FP32_KAHAN, abi.HBT_DIRECT_FP64):
            phi = torch.empty(len(c["x"]), dtype=torch.float64, device=DEV)
            torch.cuda.synchronize()
            abi.check(U.lib.hbt_direct_potential(U.ctx, len(seg) - 1, seg.data_ptr(), *p, mode, phi.data_ptr()),
                      "hbt_direct_potential")
            out.append(phi)
        return out
    if kind == "props":
        q = U.properties_device(state["h"], state["out"])
        return {f: np.ascontiguousarray(q[f]) for f in abi.PROPS_FIELDS}
    if kind == "mask":
        subs, grp, n = state["subs"], state["grp"], len(state["cols"]["id"])
        out = torch.full((n,), -1, dtype=torch.int64, device=DEV)
        kept = np.zeros(len(subs), np.int64)
        torch.cuda.synchronize()
        abi.check(U.lib.hbt_mask_subhalos(U.ctx, ctypes.byref(state["ps"]), subs.ctypes.data, grp.ctypes.data, None,
                                          len(subs), out.data_ptr(), kept.ctypes.data), "hbt_mask_subhalos")
        return dict(lists=out, kept=kept)
    subs, out, _ = U.merge_device(state["hm"], state["subs"], state["grp"], out=state["out"])
    return dict(_split_host(subs), lists=out)


# ---- what a pass cannot do without ----------------------------------------------

def _unbind_work(counts, listed_as=0):
    """Columns (40 B) read and list entries (12 B) written once per particle,
    records read and written; about two evaluations per particle (the full pass
    and one over what it kept) of 11 flops per summed source and 10 per opened
    node, whose numbers grow with the logarithm of the list (measured: about
    460 and 96 per evaluation over the power law, mostly lists of 1e4 .. 2e5)."""
    c = np.asarray(counts, np.float64)
    sources = np.minimum(c, 80.0 * np.log(1.0 + c / 80.0))
    return dict(bytes=float(c.sum() * (52 + listed_as) + 480 * len(c)), flops=float((2 * c * (13 * sources + 20)).sum()))


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "one":
        return _unbind_work([1.2 * n])
    if kind == "batch":
        return _unbind_work((1.2 if case["law"] == "power" else 1.15) * _counts(n, case["law"]))
    if kind == "share":
        # the list's IDs, and a tenth more particles in the snapshot
        return _unbind_work(1.2 * _counts(n, "power"), listed_as=12)
    if kind == "nested":
        return _unbind_work([n] + [n / 400.0] * case["nsat"])
    if kind == "tree":
        s = min(1.2 * n, 80.0 * math.log(1.0 + 1.2 * n / 80.0))
        return dict(bytes=1.2 * n * 24, flops=1.2 * n * (13 * s + 20))
    if kind == "pairs":
        c = 1.15 * _counts(n, "small").astype(np.float64)
        return dict(bytes=float(3 * 24 * c.sum()), flops=float(3 * 11 * (c * c).sum()))
    if kind == "props":
        c = float(_counts(n, "power").sum())
        return dict(bytes=24 * c + 320 * n, flops=60 * c)
    if kind == "mask":
        return dict(bytes=16 * 4000.0 * n, flops=0)
    return dict(bytes=60 * 7800.0 * n, flops=4.3e6 * n / 300 * 3000)


# ---- the values in 64 bits -------------------------------------------------------

def _pair_sum(t, s, m, eps, periodic):
    """Softened specific potentials of targets t from sources s (own terms
    included, worth -2.8 m / h each), float64."""
    h = 2.8 * eps
    step = max(1, int(4e7) // len(s))
    out = torch.empty(len(t), device=DEV, dtype=torch.float64)
    for i in range(0, len(t), step):
        r2 = torch.zeros(len(t[i:i + step]), len(s), device=DEV, dtype=torch.float64)
        for j in range(3):
            d = s[None, :, j] - t[i:i + step, None, j]
            if periodic:
                d = d - BOX * torch.round(d / BOX)
            r2 += d * d
        r = r2.sqrt()
        u = r / h
        near = torch.where(u < 0.5, -2.8 + u * u * (16.0 / 3 + u * u * (6.4 * u - 9.6)),
                           -3.2 + (1.0 / 15) / u.clamp(min=0.25) + u * u * (32.0 / 3 + u * (-16.0 + u * (9.6 - u * 32.0 / 15))))
        out[i:i + step] = torch.where(u < 1.0, near / h, -1.0 / r.clamp(min=0.5 * h)) @ m
    return out


def _self_removed(cols, eps, periodic, lo, hi):
    p = torch.stack([cols[k][lo:hi] for k in "xyz"], 1).double()
    m = cols["mass"][lo:hi].double()
    return G * (_pair_sum(p, p, m, eps, periodic) + m / eps)


def _exact_props(case, g):
    cols, subs, out_index = _props_inputs(case, g)
    n = len(subs)
    nb = torch.from_numpy(subs["nbound"].copy()).to(DEV)
    off = torch.from_numpy(subs["offset"].copy()).to(DEV)
    own = torch.repeat_interleave(torch.arange(n, device=DEV), nb)
    start = torch.cumsum(nb, 0) - nb
    rank = torch.arange(len(own), device=DEV) - start[own]
    at = out_index[off[own] + rank]
    centre = torch.from_numpy(subs["mostbound_pos"].copy()).to(DEV).double()
    d = torch.stack([cols[k][at] for k in "xyz"], 1).double() - centre[own]
    d = d - BOX * torch.round(d / BOX)
    m = float(np.float32(MASS))
    r = d.norm(dim=1)
    order = torch.argsort(r, stable=True)
    order = order[torch.argsort(own[order], stable=True)]  # by subhalo, then radius; `rank` counts in it
    rs = r[order]
    mass = m * (rank + 1).double()
    rr = rs.clamp(min=0.5)
    v = mass / rr
    big = nb > 1
    vmax = torch.zeros(n, device=DEV, dtype=torch.float64).scatter_reduce(0, own, v, "amax")
    at_max = torch.full((n,), len(own), device=DEV).scatter_reduce(
        0, own, torch.where(v == vmax[own], torch.arange(len(own), device=DEV), len(own)), "amin")
    rho = 200.0 * PROPS_HZ ** 2 / 2.0 / G
    so = torch.full((n,), -1, device=DEV).scatter_reduce(0, own, torch.where(mass > rho * rr ** 3, rank, -1), "amax")
    pick = lambda i: torch.where(big, rr[(start + i).clamp(max=len(own) - 1)], 0.0)  # noqa: E731
    m200 = torch.where(big, m * (so + 1).double(), 0.0)
    w = torch.where(rank > 0, m, 0.0)
    r2 = (r * r).clamp(min=1e-300)
    mb = torch.from_numpy(subs["mbound"].astype(np.float64)).to(DEV).clamp(min=1e-300)
    tensors = []
    for per in (w, w / r2):
        t = torch.stack([per * d[:, a] * d[:, b] for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))], 1)
        t = torch.zeros(n, 6, device=DEV, dtype=torch.float64).index_add_(0, own, t) / mb[:, None]
        tensors.append(torch.where(big[:, None], t, 0.0))
    vphys = torch.where(big, (vmax * G).sqrt(), 0.0)
    return dict(rmax_comoving=torch.where(big, rr[at_max.clamp(max=len(own) - 1)], 0.0), vmax_physical=vphys,
                rhalf_comoving=pick(nb // 2), r2sigma_comoving=pick((nb.double() * 0.955).long()),
                bound_r200crit_comoving=(m200 / rho) ** (1.0 / 3), bound_m200crit=m200,
                last_max_vmax_physical=vphys, snapshot_index_of_last_max_vmax=None,
                inertial_tensor=tensors[0], inertial_tensor_weighted=tensors[1])


def exact(case, seed):
    """In 64 bits: pair sums for the potentials (the tree's differ from them by
    its opening angle), profiles and shapes.  An unbinding has no such value:
    its energies are the tree's, in a frame that depends on every cut before."""
    kind = case["kind"]
    if kind == "tree":
        cols = _halo_columns(case, _gen(seed))
        n = len(cols["x"])
        return _self_removed(cols, 0.5, case["periodic"], 0, n) if n <= 150_000 else None
    if kind == "pairs":
        counts, cols = _pairs_inputs(case, _gen(seed))
        if (counts.astype(np.float64) ** 2).sum() > 3e10:
            return None
        ends = np.cumsum(counts)
        phi = torch.cat([_self_removed(cols, 0.5, True, e - c, e) for c, e in zip(counts.tolist(), ends.tolist())])
        return [phi, phi, phi]
    if kind == "props":
        return _exact_props(case, _gen(seed))
    return None
