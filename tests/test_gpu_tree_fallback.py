"""Barnes-Hut lists where some groups open more nodes than their table of the
opening pool holds and are left to the depth-first walk, the others not, array
for array against the host builder."""
import numpy as np
import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu


def sheet(n, sparse, seed):
    """n particles on a sheet against the face x = 0.5 of the cells that hold a
    few particles each: those groups' cells touch every node of the sheet, so that
    they open them all, the sheet's own groups only the near ones."""
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3))
    x[:, 0] = 0.5 - 1e-5 * x[:, 0]
    far = rng.random((sparse, 3))
    far[:, 0] = 0.51 + 0.48 * far[:, 0]
    far[:2] = [[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]]  # the box
    return np.concatenate([x, far])


# a table holds 16384 opened nodes, below theta of about 0.2 65536
@pytest.mark.parametrize("n,sparse,ncrit,nleaf,theta", [
    (150000, 30, 64, 1, 0.5),     # the sparse groups run out
    (40000, 30, 64, 1, 0.5),      # they do not
    (60000, 300, 64, 1, 0.4),
    (90000, 40, 500, 1, 0.19),    # the larger table
    (400000, 40, 2000, 1, 0.17),  # which runs out
])
def test_bh_lists_of_groups_that_run_out(n, sparse, ncrit, nleaf, theta):
    import pgamd
    x = sheet(n, sparse, n + sparse)
    m = np.random.default_rng(n).uniform(0.5, 1.5, len(x)) / len(x)
    h = pgamd.bh_lists(x, m, theta, ncrit, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), len(x), theta, ncrit, nleaf), True)


# at the ends of what takes a pool at all: theta so small that most groups would
# open more than a table holds, with more and with fewer nodes than that
@pytest.mark.parametrize("n,ncrit,nleaf,theta", [
    (60000, 3000, 1, 0.02), (30000, 3000, 1, 0.02), (60000, 3000, 1, 0.09), (20000, 64, 1, 1e-150),
])
def test_bh_lists_of_small_opening_angles(n, ncrit, nleaf, theta):
    import pgamd
    m, x = ics.hernquist(n, n)
    if theta < 1e-9:
        x, m = x[:3000], m[:3000]
    h = pgamd.bh_lists(x, m, theta, ncrit, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), len(x), theta, ncrit, nleaf), True)
