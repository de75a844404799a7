"""The counted work of the unbinding's sorts against its definition."""
import numpy as np
import pytest

from hbtplus_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,levels", [(700, None), (2000, 0), (3000, 1), (9000, 1), (40000, 2)])
def test_sort_bytes_of_one_pass(gpu, n, levels):
    """one list of particles so heavy that its first pass binds them all and
    converges: n sources' digits and n energies are sorted, in runs of 2,048 (one: no merge level; two: one
    level of pairs; more, alone on the card: 16 runs at a level).  Lists of up to 1,024
    sort inside their own launches and count nothing"""
    cat = synth.config1(seed=45, n_nfw=n - n // 6, n_cont=n // 6)
    cat.cols["mass"] *= np.float32(1e6)
    U = gpu(cat.params)
    U.profile(2)
    rec = U.unbind_batch(cat)[0]
    got = U.profile_sorts()
    U.profile(0)
    assert rec["n_iter"][0] == 1 and rec["list_len"][0] == n and rec["status"][0] == abi.HBT_STATUS_CONVERGED
    if levels is None:
        assert (got["elements"], got["element_levels"], got["bytes"]) == (0, 0, 0)
    else:
        assert (got["elements"], got["element_levels"]) == (2 * n, 2 * n * levels)
        assert got["bytes"] == n * ((36 + 24 * levels) + (20 + 24 * levels if levels else 12))
