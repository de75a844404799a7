"""Kernels at the sizes where they can go wrong: remainders and edges of tiles
and waves, smallest and largest of a form's range, values that take its other
branches, against the CPU oracle."""
import numpy as np
import pytest

import oracle
from hbtplus_amd import abi, synth
from helpers import assert_exact, assert_tolerant
from test_gpu_props import assert_props

pytestmark = pytest.mark.gpu

U53, U24 = 2.0 ** -53, 2.0 ** -24


def _pair_sums_of_float_separations(p, seg, pos, m):
    """The pair sums in double over separations rounded and wrapped in float32,
    as the FP32 modes form them."""
    out = np.zeros(int(seg[-1]))
    h, box, half = 2.8 * float(p["softening"][0]), np.float32(p["box_size"][0]), np.float32(p["box_size"][0] / 2)
    for lo, hi in zip(seg[:-1], seg[1:]):
        d = pos[None, lo:hi, :] - pos[lo:hi, None, :]
        assert d.dtype == np.float32
        if p["periodic"][0]:
            d = np.where(d > half, d - box, np.where(d < -half, d + box, d))
        r = np.sqrt((d.astype(np.float64) ** 2).sum(-1))
        u = r / h
        safe = np.maximum(u, 0.5)
        spline = np.where(u < 0.5, -2.8 + u * u * (16 / 3 + u * u * (6.4 * u - 9.6)),
                          -3.2 + 1 / (15 * safe) + u * u * (32 / 3 + u * (-16 + u * (9.6 - 32 / 15 * u)))) / h
        t = np.where(u < 1, spline, -1 / np.maximum(r, h)) * m[None, lo:hi].astype(np.float64)
        np.fill_diagonal(t, 0)
        out[lo:hi] = t.sum(1)
    return out * float(p["G"][0])


@pytest.mark.parametrize("where", ["inside", "across_a_face", "not_periodic"])
def test_direct_potential_sizes(gpu, where):
    """group sizes around the wave (64) and the chunk (256) and the unrolled
    four; groups inside the box, split by a face (wrapped chunks) and without a
    box; coincident particles.  All terms have one sign, so a sum of n terms of
    up to 16 roundings each is within n + 16 roundings of the exact one: of the
    oracle's for FP64, for FP32 of the double sum over float separations"""
    sizes = [1, 2, 3, 4, 5, 63, 64, 65, 127, 255, 256, 257, 511, 513, 1023, 1030]
    rng = np.random.default_rng(31)
    seg = np.concatenate([[0], np.cumsum(sizes)])
    box = 1.0e4
    pos = rng.normal(size=(seg[-1], 3)) * 20.0 + {"inside": box / 2, "across_a_face": 0.0, "not_periodic": 0.0}[where]
    pos[seg[5] + 1] = pos[seg[5]]  # a coincident pair, and pairs inside the softening length
    pos[seg[8]:seg[8] + 10] = pos[seg[8]] + rng.normal(size=(10, 3)) * 0.3
    pos = (pos % box if where != "not_periodic" else pos).astype(np.float32)
    x, y, z = (pos[:, j].copy() for j in range(3))
    m = rng.uniform(1e-5, 2e-4, len(x)).astype(np.float32)
    p = abi.make_params(periodic=int(where != "not_periodic"), box_size=box)
    U = gpu(p)
    refs = {abi.HBT_DIRECT_FP64: oracle.direct_potential(p, seg, x, y, z, m, abi.HBT_DIRECT_FP64)}
    refs[abi.HBT_DIRECT_FP32] = refs[abi.HBT_DIRECT_FP32_KAHAN] = _pair_sums_of_float_separations(p, seg, pos, m)
    n = np.repeat(sizes, sizes).astype(np.float64)
    for mode, ref in refs.items():
        got = U.direct_potential(seg, x, y, z, m, mode)
        lone = n == 1
        assert np.all(got[lone] == 0) and np.all(ref[lone] == 0)
        rel = np.abs(got[~lone] / ref[~lone] - 1)
        assert np.all(rel <= (n[~lone] + 16) * (U53 if mode == abi.HBT_DIRECT_FP64 else U24)), (mode, rel.max())


@pytest.mark.parametrize("hz,periodic", [(0.0, 0), (0.1, 1)])
def test_properties_sizes(gpu, hz, periodic):
    """bound lists of 0 to 3 entries and around the wave, the block and the
    tile: profiles bit for bit, shapes within 2 ulps of the oracle's"""
    sizes = [0, 1, 2, 3, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2049, 5000]
    rng = np.random.default_rng(37)
    n = int(np.sum(sizes))
    pos = rng.normal(size=(n, 3)) * 30.0 + (0.0 if periodic else 500.0)
    cols = {k: (pos[:, j] % 1000.0).astype(np.float32) for j, k in enumerate("xyz")}
    for k in ("vx", "vy", "vz"):
        cols[k] = rng.normal(size=n).astype(np.float32)
    cols.update(id=np.arange(n, dtype=np.int64), mass=rng.uniform(1e-4, 2e-4, n).astype(np.float32),
                type=np.ones(n, np.int32))
    subs = np.zeros(len(sizes), abi.SUB_DTYPE)
    subs["count"] = subs["nbound"] = sizes
    subs["parent"] = -1
    subs["offset"] = subs["out_offset"] = np.cumsum(sizes) - sizes
    index = rng.permutation(n).astype(np.int64)  # lists of scattered columns
    for s in subs:
        l = index[s["out_offset"]:s["out_offset"] + s["nbound"]]
        if len(l):
            s["mostbound_pos"] = [cols[k][l[0]] for k in "xyz"]
            s["mbound"] = cols["mass"][l].astype(np.float64).sum()
    p = abi.make_params(hz=hz, periodic=periodic, box_size=1000.0)
    U = gpu(p)
    cat = synth.Catalogue(cols, subs, p)
    h = U.upload(cat)
    got = U.properties_device(h, (U._dev(subs.view(np.uint8)), U._dev(index), None))
    assert_props(oracle.subhalo_properties(p, cols, subs, index, np.zeros(len(subs), abi.PROPS_DTYPE)), got)


@pytest.mark.parametrize("n_src", [1, 2, 17, 1024, 5000])
@pytest.mark.parametrize("periodic", [0, 1])
def test_tree_potential_target_orders(gpu, n_src, periodic):
    """the counting sort of the targets: fewer and more targets than a wave, a
    block or the sources, all in one place, outside the sources' cube, across a
    face; one that is not a number spoils nobody else's wrap.  REPLAY bit for
    bit, FAST within its 1e-5 of the oracle"""
    rng = np.random.default_rng(n_src)
    box = 1.0e4
    sp = (rng.normal(size=(n_src, 3)) * 25.0 + 60.0) % box
    src = tuple(sp[:, j].astype(np.float32) for j in range(3)) + (rng.uniform(1e-4, 2e-4, n_src).astype(np.float32),)
    for kind, nt in (("near", 1), ("near", 63), ("near", 257), ("same", 3000), ("far", 130), ("edge", 700), ("nan", 65)):
        tp = rng.normal(size=(nt, 3)) * 30.0 + 60.0
        if kind == "same":
            tp[:] = tp[0]
        elif kind == "far":
            tp += rng.uniform(-3000, 3000, size=(nt, 3))
        elif kind == "edge":
            tp -= 110.0
        tp = tp % box if periodic else tp
        tgt = [tp[:, j].astype(np.float32) for j in range(3)]
        if kind == "nan":
            tgt[1][7] = np.nan
        for prec in (abi.HBT_PREC_REPLAY, abi.HBT_PREC_FAST):
            p = abi.make_params(periodic=periodic, box_size=box, precision=prec)
            ref = oracle.tree_potential(p, src, tgt, None)
            got = gpu(p).tree_potential(src, tgt, None)
            ok = ~np.isnan(tgt[1])  # (FAST takes an undefined distance as 0, the oracle does not)
            assert np.all(np.isfinite(ref[ok])), (kind, nt)
            if prec == abi.HBT_PREC_REPLAY:
                assert np.array_equal(ref[ok], got[ok]), (kind, nt)
            else:
                assert np.abs(got[ok] / ref[ok] - 1).max() < 1e-5, (kind, nt)


@pytest.mark.parametrize("at_edges", [False, True])
def test_shared_walk_changes_no_bit(gpu, at_edges):
    """a level of more than 6,144 chunks of targets is walked one wave to a
    chunk, each of its subhalos alone by up to 16 waves sharing the items: the
    FP64 sums are exact for terms this far apart (masses over a factor of 30,
    lists up to 20,000), so records, lists and energies agree byte for byte"""
    cat = synth.config2(seed=81, nsub=2600, hi=2.0e4, at_edges=at_edges)
    assert np.sum((cat.subs["count"] + 63) // 64) > 6144
    cat.cols["mass"] = (1e-4 * np.random.default_rng(5).uniform(1, 30, cat.n_particles)).astype(np.float32)
    U = gpu(cat.params)
    for a, b in zip(U.unbind_batch(cat), U.unbind_batch(cat, plain=True)):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("coincident", [False, True])
def test_tree_forms(gpu, coincident):
    """a list's first n particles at the sizes where its trees change form: one
    wave (64, 256), one workgroup (1,024), tiles, super-tiles (65,536); REPLAY
    against the oracle bit for bit, and where runs of particles share one place
    (whole subtrees at the resolution floor, whose inner order the reference
    draws at random) its tolerant criteria"""
    base = synth.config1(seed=93, n_nfw=56600, n_cont=10000)
    if coincident:
        for c in ("x", "y", "z"):
            base.cols[c][1:2001:2] = base.cols[c][:2000:2]
            base.cols[c][4000:4300] = base.cols[c][4000]
    sizes = [2, 3, 7, 62, 64, 65, 130, 254, 256, 257, 700, 1022, 1024, 1025, 2048, 2049, 5000, 65536, 65537, 66600]
    cols = {c: np.concatenate([a[:n] for n in sizes]) for c, a in base.cols.items()}
    cols["id"] = np.arange(sum(sizes), dtype=np.int64)
    cols["mass"] *= np.repeat(66600 / np.float32(sizes), sizes)  # each list as bound as the whole
    subs = np.repeat(base.subs[:1], len(sizes))
    subs["count"] = subs["nbound_prev"] = sizes
    subs["offset"] = np.cumsum([0] + sizes[:-1])
    p = base.params.copy()
    p["precision"] = abi.HBT_PREC_REPLAY
    cat = synth.Catalogue(cols, subs, p, "tree forms")
    ref = oracle.unbind_batch(cat, nthreads=16)
    got = gpu(p).unbind_batch(cat)
    if coincident:
        assert_tolerant(ref, got)
    else:
        assert_exact(ref, got)
    for a, b in zip(got, gpu(p).unbind_batch(cat, plain=True)):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("prec", [abi.HBT_PREC_REPLAY, abi.HBT_PREC_FAST])
@pytest.mark.parametrize("refine", [0, 1])
def test_one_tile_passes_with_a_sample(gpu, prec, refine):
    """lists of up to a few tiles with a sample of 20: most are shuffled, their
    trees hold 20 sources, and with the refinement their outputs wait for it;
    REPLAY equals the oracle, FAST meets the band rule, and the captured pass
    sequence (no list swap) and the plain form give the batched bytes"""
    cat = synth.config2(seed=95, nsub=400, hi=3000)
    cat.params["max_sample_size"] = 20
    cat.params["refine_mostbound_particle"] = refine
    cat.params["precision"] = prec
    ref = oracle.unbind_batch(cat, nthreads=8, rand_state={"seed": 1, "draws": 0})
    U = gpu(cat.params)
    got = U.unbind_batch(cat)
    if prec == abi.HBT_PREC_REPLAY:
        assert_exact(ref, got)
    else:
        assert_tolerant(ref, got, refined=20 if refine else 0)
    for form in ("graph", "plain"):
        U.set_rand_state(1, 0)
        t = U.get_tuning()
        t["use_graph"] = int(form == "graph")
        U.set_tuning(t)
        for a, b in zip(got, U.unbind_batch(cat, plain=form == "plain")):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), form


@pytest.mark.parametrize("softening", [0.0108, 0.5])
def test_digit_sorts(gpu, softening):
    """octant digits of 19 depths leave a word no room for the place in the
    run, and are sorted as pairs, those of 13 as words; a few equal digits (pairs
    of sources closer than the smallest cell) are ordered by their values.
    REPLAY against the oracle bit for bit, at the sizes of each sort"""
    base = synth.config1(seed=97, n_nfw=8000, n_cont=1000)
    sizes = [3, 60, 250, 1000, 2000, 2100, 9000]
    cols = {c: np.concatenate([a[:n] for n in sizes]) for c, a in base.cols.items()}
    cols["id"] = np.arange(sum(sizes), dtype=np.int64)
    cols["mass"] *= np.repeat(9000 / np.float32(sizes), sizes)
    subs = np.repeat(base.subs[:1], len(sizes))
    subs["count"] = subs["nbound_prev"] = sizes
    subs["offset"] = np.cumsum([0] + sizes[:-1])
    p = base.params.copy()
    p["precision"], p["softening"] = abi.HBT_PREC_REPLAY, softening
    cat = synth.Catalogue(cols, subs, p, "digit sorts")
    assert_exact(oracle.unbind_batch(cat, nthreads=8), gpu(p).unbind_batch(cat))


def test_single_call_staging(gpu):
    """the single call sends its columns through pinned memory up to 131,072
    particles and straight from the caller's arrays above: both give the batched
    bytes, as do a list of one particle and one without types; a type out of range
    and a missing column are errors either way"""
    base = synth.config1(seed=98, n_nfw=120000, n_cont=11073)
    U = gpu(base.params)
    for n in (1, 131072, 131073):
        for types in (True, False):
            cols = {c: a[:n] for c, a in base.cols.items() if types or c != "type"}
            sub = base.subs[:1].copy()
            sub["count"] = n
            # (a batch of one list unbinds one that had a single particle as an orphan)
            sub["nbound_prev"] = max(n, 2)
            rec, idx, e = U.unbind_one(cols, sub)
            full = dict(cols, type=np.ones(n, np.int32))
            r, i, f = U.unbind_batch(synth.Catalogue(full, sub, base.params, "one"))
            assert np.array_equal(i, idx) and np.array_equal(f.view(np.uint32), e.view(np.uint32))
            assert np.array_equal(r.view(np.uint8), rec.view(np.uint8))
        bad = dict(base.cols, type=np.full(n, 6, np.int32))
        with pytest.raises(RuntimeError, match="particle types outside"):
            U.unbind_one({c: a[:n] for c, a in bad.items()}, sub)
        with pytest.raises(RuntimeError, match="null argument"):
            U.unbind_one({c: a[:n] for c, a in base.cols.items() if c != "vx"}, sub)


@pytest.mark.parametrize("sizes", [(4096, 4097, 8193, 32767, 32768, 32769, 60000), (2049, 4097, 5000, 70000)])
def test_ranked_runs(gpu, sizes):
    """sorts of 3 runs of 2,048 and more in a launch of few tiles rank their
    elements, 16 runs at a level, instead of merging pairs: lists alone (ranked;
    one level up to 32,768), many together (merged) and a few together (ranked
    in one launch) give the same bytes; every 97th particle shares its place
    with the one before, so equal digits fall into one run and into several"""
    n = max(sizes)
    base = synth.config1(seed=99, n_nfw=n - n // 6, n_cont=n // 6)
    for c in ("x", "y", "z"):
        base.cols[c][1:n:97] = base.cols[c][0:n - 1:97][:len(base.cols[c][1:n:97])]
        base.cols[c][5::511] = base.cols[c][5]
    cols = {c: np.concatenate([a[:m] for m in sizes]) for c, a in base.cols.items()}
    cols["id"] = np.arange(sum(sizes), dtype=np.int64)
    cols["mass"] *= np.repeat(n / np.float32(sizes), sizes)
    subs = np.repeat(base.subs[:1], len(sizes))
    subs["count"] = subs["nbound_prev"] = sizes
    subs["offset"] = np.cumsum((0,) + sizes[:-1])
    cat = synth.Catalogue(cols, subs, base.params, "ranked runs")
    U = gpu(cat.params)
    got = U.unbind_batch(cat)
    assert (got[0]["status"] == abi.HBT_STATUS_CONVERGED).all()
    assert_tolerant(oracle.unbind_batch(cat, nthreads=8), got)
    for a, b in zip(got, U.unbind_batch(cat, plain=True)):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("ids", ["mixed", "one", "high_bits"])
def test_mask_claims(gpu, ids):
    """groups of 1 to 9,000 entries in several subhalos: first claims in a table
    of one workgroup (up to 1,024 and 8,192 entries) and by sorting; IDs repeated
    in and across lists, one ID alone, IDs that differ in their high bits only"""
    rng = np.random.default_rng(41)
    sizes = [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2049, 8191, 8192, 8193, 9000]
    counts, grp, parent, pool = [], [], [], []
    for g, n in enumerate(sizes):
        cuts = np.sort(rng.integers(0, n + 1, min(n - 1, 6)))
        part = np.diff(np.concatenate([[0], cuts, [n]]))  # some lists empty
        first = len(counts)
        counts += list(part)
        grp += [g] * len(part)
        parent += [-1] + [int(rng.integers(first, first + i)) if i % 2 else -1 for i in range(1, len(part))]
        pool.append(rng.integers(0, max(1, n * 2 // 3), n))
    ident = np.concatenate(pool).astype(np.int64)
    if ids == "mixed":
        ident = np.where(rng.random(len(ident)) < 0.1, np.int64(-1), ident - 500)
    elif ids == "one":
        ident[:] = 7
    else:
        ident = (ident << 48) ^ np.int64(1)
    subs = np.zeros(len(counts), abi.SUB_DTYPE)
    subs["count"] = subs["nbound_prev"] = counts
    subs["offset"] = np.cumsum([0] + counts[:-1])
    subs["parent"] = parent
    subs["nbound_prev"][5::9] = 1  # claim nothing
    n = len(ident)
    cols = {k: np.zeros(n, np.float32) for k in ("x", "y", "z", "vx", "vy", "vz", "mass")}
    cols.update(id=ident, type=np.ones(n, np.int32))
    grp = np.array(grp, np.int64)
    out, cnt = gpu(abi.make_params()).mask_subhalos(cols, subs, grp)
    ref_out, ref_cnt = oracle.mask_subhalos(cols, subs, grp)
    assert np.array_equal(cnt, ref_cnt)
    for o, c in zip(subs["offset"], cnt):
        assert np.array_equal(out[o:o + c], ref_out[o:o + c])
