"""Pair sums of groups of at most 64 particles, a wave each, alone and among
larger ones, through both entry points."""
import ctypes

import numpy as np
import pytest

import oracle
from hbtplus_amd import abi
from test_gpu_kernels import U24, U53, _pair_sums_of_float_separations

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("others", ["alone", "with_larger"])
@pytest.mark.parametrize("where", ["inside", "across_a_face", "a_quarter_box_wide", "not_periodic"])
def test_groups_of_up_to_a_wave(gpu, others, where):
    """sizes 0 to 64, one of each and many of one; coincident particles; groups
    wide enough to wrap pairs.  A sum of n terms of one sign, of up to 16 roundings
    each, is within n + 16 roundings of the exact one; the entry point that
    allocates nothing gives the same bits"""
    import torch

    sizes = list(range(65)) + [5] * 1100 + ([65, 300, 0, 1025, 64] if others == "with_larger" else [])
    rng = np.random.default_rng(len(sizes))
    np.random.default_rng(7).shuffle(sizes)
    seg = np.concatenate([[0], np.cumsum(sizes)])
    box = 1.0e4
    width, at = {"inside": (20.0, box / 2), "across_a_face": (20.0, 0.0), "a_quarter_box_wide": (box / 8, box / 2),
                 "not_periodic": (20.0, 0.0)}[where]
    pos = rng.normal(size=(seg[-1], 3)) * width + at
    big = int(np.argmax(np.array(sizes) == 40))
    pos[seg[big] + 1] = pos[seg[big]]
    pos[seg[big] + 3:seg[big] + 9] = pos[seg[big]] + rng.normal(size=(6, 3)) * 0.3
    pos = (pos % box if where != "not_periodic" else pos).astype(np.float32)
    x, y, z = (pos[:, j].copy() for j in range(3))
    m = rng.uniform(1e-5, 2e-4, len(x)).astype(np.float32)
    p = abi.make_params(periodic=int(where != "not_periodic"), box_size=box)
    U = gpu(p)
    refs = {abi.HBT_DIRECT_FP64: oracle.direct_potential(p, seg, x, y, z, m, abi.HBT_DIRECT_FP64)}
    refs[abi.HBT_DIRECT_FP32] = refs[abi.HBT_DIRECT_FP32_KAHAN] = _pair_sums_of_float_separations(p, seg, pos, m)
    n = np.repeat(sizes, sizes).astype(np.float64)
    dev = [torch.from_numpy(a).cuda() for a in (x, y, z, m)]
    off = torch.from_numpy(seg.astype(np.int64)).cuda()
    for mode, ref in refs.items():
        got = U.direct_potential(seg, x, y, z, m, mode)
        lone = n == 1
        assert np.all(got[lone] == 0)
        rel = np.abs(got[~lone] / ref[~lone] - 1)
        assert np.all(rel <= (n[~lone] + 16) * (U53 if mode == abi.HBT_DIRECT_FP64 else U24)), (mode, rel.max())
        out = torch.zeros(len(x), dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        fn = U.lib.hbt_direct_potential_noalloc
        abi.check(fn(U.ctx, ctypes.c_int64(len(sizes)), *[ctypes.c_void_p(t.data_ptr()) for t in (off, *dev)], mode,
                     ctypes.c_void_p(out.data_ptr())), "hbt_direct_potential_noalloc")
        assert np.array_equal(out.cpu().numpy().view(np.uint64), got.view(np.uint64)), mode
