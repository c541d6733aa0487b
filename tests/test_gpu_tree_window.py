"""GPU list builds with groups of thousands of particles up to one group of all,
array for array against the host builder; the work of a build depends on the
particles, not on how far the group size lies above their number."""
import time

import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu

LARGEST = 2 ** 31 - 1


# the sliding maximum: 1025 places in LDS, then doubled: 2050, 4100, ...
@pytest.mark.parametrize("n,ncrit", [
    (9001, 1024), (9001, 1025), (9001, 2049), (9001, 2050), (9001, 4099), (9001, 4100),
    (9001, 8999), (9001, 9000), (9001, 9001), (9001, 9002), (9001, LARGEST), (1, LARGEST),
    (600, LARGEST - 1), (300000, 70000),
])
def test_treepm_lists_of_large_groups(n, ncrit):
    import pgamd
    _, x = ics.clumpy_box(n, n + 3, nclump=3, sigma=0.003)
    h = pgamd.treepm_lists(x, 0.07, ncrit)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), n, 0.07, ncrit), False)


@pytest.mark.parametrize("n,ncrit,nleaf", [
    (6000, 3000, 2050), (6000, LARGEST, 1026), (6000, LARGEST, LARGEST), (6000, 5999, 6001),
])
def test_bh_lists_of_large_groups_and_leaves(n, ncrit, nleaf):
    import pgamd
    m, x = ics.hernquist(n, n)
    h = pgamd.bh_lists(x, m, 0.5, ncrit, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, 0.5, ncrit, nleaf), True)


def test_build_time_does_not_grow_with_the_group_size():
    import pgamd
    n = 4096
    _, x = ics.clumpy_box(n, 1)
    d_x = dev(x)

    def best(ncrit):
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            pgamd.DevLists.treepm(d_x.data_ptr(), n, 0.07, ncrit).free()
            t.append(time.perf_counter() - t0)
        return min(t)

    # one group either way: the same work, but for the noise of a build of 0.4 ms
    assert best(1 << 24) < 5 * best(n)
