"""hbt_tree_potential at the sizes where its walk changes form, and trees beyond
the reach of 32-bit byte offsets (2^27 items of 32 bytes)."""
import numpy as np
import pytest

import oracle
from hbtplus_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tgt", [300, 140_000])
def test_tree_of_more_than_2_27_items(gpu, n_tgt):
    """100 million sources of mass 1e-30 fill a corner of the cube, before a halo
    of 5,000 in the tree's order, whose items therefore lie beyond 2^27 (about 1.45
    items to a source).  The halo's targets accept the corner as a node or a few,
    terms of 1e-23 that leave sums of 0.1 and more as they are, so the potentials are
    those of the halo and one corner source that spans the same cube: REPLAY bit for
    bit, FAST and FP32 within their 1e-5 of the oracle"""
    import torch

    from hbtplus_amd.device import GpuUnbinder

    rng = np.random.default_rng(61)
    n_fill, n_halo = 100_000_000, 5000
    halo = (7.5 + 0.1 * rng.standard_normal((n_halo, 3))).clip(7.0, 8.0).astype(np.float32)
    halo[-1] = 8.0  # the cube's far corner; the fill's first source is the near one
    mass = rng.uniform(1e-4, 2e-4, n_halo).astype(np.float32)
    tgt = (7.5 + 0.15 * rng.standard_normal((n_tgt, 3))).clip(6.8, 8.2).astype(np.float32)
    fill = torch.rand(3, n_fill, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(7))
    fill[:, 0] = 0.0
    src = [torch.cat([fill[j], torch.from_numpy(halo[:, j].copy()).cuda()]) for j in range(3)]
    src.append(torch.cat([torch.full((n_fill,), 1e-30, device="cuda:0"), torch.from_numpy(mass).cuda()]))
    del fill
    t = [torch.from_numpy(tgt[:, j].copy()).cuda() for j in range(3)]
    out = torch.empty(n_tgt, dtype=torch.float64, device="cuda:0")
    few = (*(np.concatenate([[np.float32(0)], halo[:, j]]) for j in range(3)),
           np.concatenate([[np.float32(1e-30)], mass]))
    check = rng.permutation(n_tgt)[:300]
    for prec in (abi.HBT_PREC_REPLAY, abi.HBT_PREC_FP32, abi.HBT_PREC_FAST):
        p = abi.make_params(softening=1e-4, open_angle=0.45, periodic=0, precision=prec)
        ref = oracle.tree_potential(p, few, tuple(tgt[check, j].copy() for j in range(3)), None)
        assert np.all(np.abs(ref) > 0.1 * float(p["G"][0]))
        with GpuUnbinder(p, device=0) as U:
            torch.cuda.synchronize()
            abi.check(U.lib.hbt_tree_potential(U.ctx, n_fill + n_halo, *[s.data_ptr() for s in src], n_tgt,
                                               *[s.data_ptr() for s in t], None, out.data_ptr()), "hbt_tree_potential")
            got = out.cpu().numpy()[check]
        if prec == abi.HBT_PREC_REPLAY:
            assert np.array_equal(ref, got)
        else:
            assert np.abs(got / ref - 1).max() < (1e-5 if prec == abi.HBT_PREC_FAST else n_halo * 2.0 ** -24)


def test_walk_group_forms_of_many_chunks(gpu):
    """a level of more than 6,144 chunks is walked by the tuned groups (smaller ones
    share their chunks whatever the groups): 8, 16, 32 and 64 lanes and groups by
    segment give the same bytes in FAST and FP32"""
    from hbtplus_amd import synth

    cat = synth.config2(seed=83, nsub=2600, hi=2.0e4)
    assert np.sum((cat.subs["count"] + 63) // 64) > 6144
    for prec in (abi.HBT_PREC_FAST, abi.HBT_PREC_FP32):
        cat.params["precision"] = prec
        U = gpu(cat.params)
        got = []
        for groups in ((16, 16, 16), (8, 8, 8), (32, 32, 32), (64, 64, 64), (64, 8, 32)):
            t = U.get_tuning()
            t["walk_group"] = groups
            t["bin_edge"] = (100, 700)
            U.set_tuning(t)
            got.append(U.unbind_batch(cat))
        for other in got[1:]:
            for x, y in zip(got[0], other):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), prec


@pytest.mark.parametrize("n_src", [1, 100, 65535, 65536])
@pytest.mark.parametrize("n_tgt", [1, 255, 257, 263_001])
def test_tree_targets_by_buckets(gpu, n_src, n_tgt):
    """targets counted by buckets of 16 sources, in LDS up to 4,096 buckets (65,535
    sources) by runs of 256 targets and more, and in memory beyond; half of the
    targets stand in one place.  Any order of the targets gives the same bits, and a
    sample of them the oracle's"""
    rng = np.random.default_rng(n_src + n_tgt)
    sp = rng.normal(size=(n_src, 3)) * 25.0 + 500.0
    src = tuple(sp[:, j].astype(np.float32) for j in range(3)) + (rng.uniform(1e-4, 2e-4, n_src).astype(np.float32),)
    tp = (rng.normal(size=(n_tgt, 3)) * 30.0 + 500.0).astype(np.float32)
    tp[rng.random(n_tgt) < 0.5] = tp[0]
    perm, some = rng.permutation(n_tgt), rng.integers(0, n_tgt, 200)
    cols = lambda a: tuple(a[:, j].copy() for j in range(3))  # noqa: E731
    for prec in (abi.HBT_PREC_REPLAY, abi.HBT_PREC_FAST):
        p = abi.make_params(periodic=1, box_size=1.0e4, precision=prec)
        U = gpu(p)
        got = U.tree_potential(src, cols(tp))
        assert np.array_equal(got[perm].view(np.uint64), U.tree_potential(src, cols(tp[perm])).view(np.uint64))
        ref = oracle.tree_potential(p, src, cols(tp[some]))
        if prec == abi.HBT_PREC_REPLAY:
            assert np.array_equal(ref, got[some])
        else:
            assert np.abs(got[some] / ref - 1).max() < 1e-5


@pytest.mark.parametrize("n_src", [1, 64, 65, 1025, 5000, 200_000])
@pytest.mark.parametrize("where", ["inside", "across_a_face", "not_periodic"])
def test_target_walks_agree(gpu, n_src, where):
    """a few targets and many of them take other forms of the walk (each lane alone,
    the targets as they came or in tree order; lanes together, by chunks of dense
    targets; a chunk shared by waves): the same target gets the same bits, in every
    precision, among the sources, beside them and far away"""
    rng = np.random.default_rng(n_src)
    box, n_tgt = 1.0e4, 140_000
    at = {"inside": 500.0, "across_a_face": 0.0, "not_periodic": 0.0}[where]
    wrap = (lambda a: (a % box).astype(np.float32)) if where != "not_periodic" else (lambda a: a.astype(np.float32))
    sp, tp = wrap(rng.normal(size=(n_src, 3)) * 25.0 + at), wrap(rng.normal(size=(n_tgt, 3)) * 30.0 + at)
    far = rng.random(n_tgt) < 0.3
    tp[far] = wrap(rng.uniform(-4000, 4000, size=(int(far.sum()), 3)) + at)
    src = tuple(sp[:, j].copy() for j in range(3)) + (rng.uniform(1e-4, 2e-4, n_src).astype(np.float32),)
    for prec in (abi.HBT_PREC_REPLAY, abi.HBT_PREC_FP32, abi.HBT_PREC_FAST):
        U = gpu(abi.make_params(periodic=int(where != "not_periodic"), box_size=box, precision=prec))
        full = U.tree_potential(src, tuple(tp[:, j].copy() for j in range(3)))
        for n in (1, 4, 70, 3000, 30000):
            some = rng.permutation(n_tgt)[:n]
            got = U.tree_potential(src, tuple(tp[some, j].copy() for j in range(3)))
            assert np.array_equal(got.view(np.uint64), full[some].view(np.uint64)), (prec, n)
