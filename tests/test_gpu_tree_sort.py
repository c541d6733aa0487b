"""The list builds' counting sort at the edges of its blocks and of the runs
of equal upper key bits, array for array against the host builder."""
import numpy as np
import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu

# 2^18 pairs and more are sorted by counting, in blocks of 4096; the last 23
# bits of the keys (positions that share 13 bits an axis) in runs of up to
# 2049, with one more by all 63 bits
SIZES = [(262143, 0), (262144, 3), (262145, 2048), (266239, 2049), (266240, 2050), (266241, 5000)]


def put_run(x, run):
    """x with `run` particles inside one cell of 2^-13, 2^-21 apart or coincident."""
    rng = np.random.default_rng(run)
    at = rng.permutation(len(x))[:run]
    x[at] = (1234 + (rng.integers(0, 256, (run, 3)) + 0.5) / 256) / 8192
    return x


# the cells' numbers take 8 bits at a cut-off of 0.2 and 17 at 0.02
@pytest.mark.parametrize("n,run,rcut", [s + (0.02,) for s in SIZES] + [(262144, 0, 0.2)])
def test_treepm_lists_sorted_by_counting(n, run, rcut):
    import pgamd
    x = put_run(np.random.default_rng(n).random((n, 3)), run)
    h = pgamd.treepm_lists(x, rcut, 64)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), n, rcut, 64), False)


# one group a particle: more groups than are ordered by counting pairs (16384)
@pytest.mark.parametrize("n,ncrit", [(16000, 1), (17000, 1), (262144, 1), (266241, 8)])
def test_bh_lists_ordered_by_cost(n, ncrit):
    import pgamd
    m, x = ics.hernquist(n, n)
    h = pgamd.bh_lists(x, m, 1.0, ncrit, 8)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, 1.0, ncrit, 8), True)


# one group a particle: counts per group in tiles of 4096 of one block, up to
# eight of them, and more; ghosts in blocks of 1024 particles
@pytest.mark.parametrize("n", [4095, 4096, 4097, 8193, 32767, 32768, 32769])
def test_treepm_lists_at_scan_edges(n):
    import pgamd
    x = np.random.default_rng(n).random((n, 3))
    h = pgamd.treepm_lists(x, 0.04, 1)
    d_x = dev(x)
    L = pgamd.DevLists.treepm(d_x.data_ptr(), n, 0.04, 1)
    assert L.info()["ngroups"] == n
    check(h, L, False)
