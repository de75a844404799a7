"""Early exits whose lists are long: orphan hosts of no or one particle that
take over their subhalos' tails."""
import numpy as np
import pytest

import oracle
from hbtplus_amd import abi, synth
from helpers import OUTPUT_FIELDS, list_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.HBT_PREC_FAST, abi.HBT_PREC_REPLAY])
def test_orphan_hosts_over_long_tails(gpu, prec):
    """hosts of 0 and 1 particles over subhalos that fall apart (particles far too
    fast to be bound), each of which leaves all of its particles but one to the host:
    lists of 1 to 4 entries, of one tile of 1,024 and one more, and of several tiles;
    a host without particles that is no orphan among them.  Records and lists,
    order included, are the oracle's"""
    nests = [(0, [3]), (1, [3]), (1, []), (0, []), (1, [1024]), (1, [1025]), (0, [1025]), (0, [1026]), (1, [60, 3000, 2]),
             (0, [70000, 5]), (1, [4100, 9000, 1500])]
    counts, parent = [], []
    for host, kids in nests:
        at = len(counts)
        counts += [host] + kids
        parent += [-1] + [at] * len(kids)
    counts, n = np.array(counts), int(np.sum(counts))
    rng = np.random.default_rng(71)
    cols = {k: (rng.normal(size=n) * 50.0 + 500.0).astype(np.float32) for k in "xyz"}
    for k in ("vx", "vy", "vz"):
        cols[k] = (rng.normal(size=n) * 1.0e5).astype(np.float32)
    cols.update(id=rng.permutation(n).astype(np.int64), mass=np.full(n, 1e-4, np.float32),
                type=rng.integers(0, 6, n).astype(np.int32))
    subs = np.zeros(len(counts), abi.SUB_DTYPE)
    subs["count"], subs["parent"] = counts, parent
    subs["offset"] = np.cumsum(counts) - counts
    subs["nbound_prev"] = np.where(subs["parent"] < 0, subs["count"], np.maximum(counts, 2))
    subs["nbound_prev"][5] = 5  # the host without particles or subhalos: no orphan
    for f in ("sink_track_id", "snapshot_index_of_death", "snapshot_index_of_sink"):
        subs[f] = -1
    cat = synth.Catalogue(cols, subs, abi.make_params(precision=prec, periodic=0), "early lists")
    ref = oracle.unbind_batch(cat)
    for plain in (False, True):
        got = gpu(cat.params).unbind_batch(cat, plain=plain)
        for f in OUTPUT_FIELDS:
            assert np.array_equal(ref[0][f], got[0][f]), f
        for s in range(len(counts)):
            assert np.array_equal(list_of(ref[0], ref[1], s), list_of(got[0], got[1], s)), s
    long = [s for s in range(len(counts)) if parent[s] < 0 and got[0]["list_len"][s] > 1024]
    assert len(long) >= 4 and (got[0]["status"][long] == abi.HBT_STATUS_EARLY).all()
