"""Moments of Barnes-Hut leaves of every small size and of leaves that the key
cannot split, bit for bit against the host builder."""
import numpy as np
import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nleaf,same", [
    (2000, 1, 0), (2000, 3, 2), (2000, 4, 3), (2001, 5, 5), (2002, 7, 9), (2003, 9, 63),
    (5000, 33, 1000), (30000, 8, 16383), (30000, 8, 16385),
])
def test_leaf_moments_at_their_remainders(n, nleaf, same):
    import pgamd
    rng = np.random.default_rng(n + same)
    _, x = ics.hernquist(n, n)
    m = rng.uniform(0.1, 1.0, n)
    for c in range(3 if same < 100 else 1):  # particles within 2^-23 of the box
        at = rng.permutation(n)[:same]
        x[at] = x[int(rng.integers(n))] + 1e-7 * rng.uniform(-1, 1, (same, 3))
    h = pgamd.bh_lists(x, m, 0.5, 64, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, 0.5, 64, nleaf), True)
