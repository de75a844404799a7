"""Tree nodes whose sources cross the edges of tiles of 1,024: a workgroup computes
up to 1,024 of a super-tile's (64 tiles) from LDS, longer lists depth by depth."""
import numpy as np
import pytest

import oracle
from hbtplus_amd import abi

LEN, TILE, DEPTH = 1024.0, 1024, 21


def nested_clusters(bulk_depth, seed):
    """64 clusters, one in each cell of depth 2 of the cube [0, 1024]: each a chain of
    cells down to bulk_depth with one source before and one behind the chain at
    every depth, the rest on distinct cells of depth 21 in its last cell.  The first
    cluster is half a tile shorter, so that every tile edge lies among a cluster's
    last"""
    rng = np.random.default_rng(seed)
    side = 2 ** (DEPTH - bulk_depth)
    pos = []
    for i in range(64):
        c, half = np.full(3, LEN / 2), LEN / 4

        def sub(c, half, digit):
            return c + half * (2.0 * ((digit >> np.arange(3)) & 1) - 1.0)

        for digit in (i >> 3, i & 7):
            c, half = sub(c, half, digit), half / 2
        for _ in range(2, bulk_depth):
            pos += [sub(c, half, 0), sub(c, half, 7)]
            c, half = sub(c, half, int(rng.integers(1, 7))), half / 2
        n = TILE - 2 * (bulk_depth - 2) - (TILE // 2 if i == 0 else 0) - (i in (0, 63))
        cell = rng.choice(side ** 3, n, replace=False)
        cell = np.stack([cell % side, cell // side % side, cell // side ** 2], 1)
        pos += list(c - 2 * half + (cell + 0.5) * (4 * half / side))
    pos += [np.zeros(3), np.full(3, LEN)]  # they span the cube
    return rng.permutation(np.array(pos)).astype(np.float32)


def crossing_nodes(pos):
    """nodes with sources on both sides of a tile edge, chains of one son left out"""
    c, half = np.full(pos.shape, LEN / 2), LEN / 2
    digits = np.zeros((len(pos), DEPTH), np.int64)
    for d in range(DEPTH):
        half /= 2
        up = pos > c
        digits[:, d] = up @ [1, 2, 4]
        c = c + np.where(up, half, -half)
    key = np.sort(digits @ 8 ** np.arange(DEPTH - 1, -1, -1))
    assert len(np.unique(key)) == len(key)  # no cell of two sources
    listed = 0
    for d in range(DEPTH):
        cell, son = key >> 3 * (DEPTH - d), key >> 3 * (DEPTH - d - 1)
        name, lo, n = np.unique(cell, return_index=True, return_counts=True)
        hi = lo + n - 1
        listed += int(np.sum((lo // TILE != hi // TILE) & (son[lo] != son[hi])))
    return listed


@pytest.mark.parametrize("bulk_depth,more", [(17, True), (12, False)])
def test_the_lists_lengths(bulk_depth, more):
    assert (crossing_nodes(nested_clusters(bulk_depth, 71)) > 1024) == more


@pytest.mark.gpu
@pytest.mark.parametrize("bulk_depth", [17, 12])
def test_crossing_nodes_of_a_super_tile(gpu, bulk_depth):
    """REPLAY equals the oracle bit for bit for targets at 3 to 6 cell sizes of every
    depth from the clusters' ends, which accept the chains' nodes"""
    pos = nested_clusters(bulk_depth, 71)
    rng = np.random.default_rng(72)
    mass = rng.uniform(0.5, 2.0, len(pos)).astype(np.float32)
    size = LEN / 2.0 ** rng.integers(2, 20, 20_000)
    away = rng.standard_normal((len(size), 3))
    away *= (rng.uniform(3, 6, len(size)) * size / np.linalg.norm(away, axis=1))[:, None]
    tgt = (pos[rng.integers(0, len(pos), len(size))] + away).astype(np.float32)
    p = abi.make_params(softening=6e-3, open_angle=0.45, periodic=0, precision=abi.HBT_PREC_REPLAY)
    src = (*(pos[:, j].copy() for j in range(3)), mass)
    to = tuple(tgt[:, j].copy() for j in range(3))
    assert np.array_equal(oracle.tree_potential(p, src, to), gpu(p).tree_potential(src, to))
