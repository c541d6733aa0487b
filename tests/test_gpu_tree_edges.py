"""GPU list builds at the edges of their blocks, windows and queues, array for
array against the host builder."""
import numpy as np
import pytest

import ics

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "src", "ioff", "icnt", "ilist", "joff", "jcnt", "jlist", "coff", "ccnt", "order")


def dev(a):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    torch.cuda.synchronize()
    return t


def check(h, L, cells):
    d = L.host()
    L.free()
    for k in FIELDS:
        np.testing.assert_array_equal(d[k], h[k], err_msg=k)
    assert d["work_pp"] == h["work_pp"] and d["work_pc"] == h["work_pc"]
    if cells:
        np.testing.assert_array_equal(d["cells"][d["clist"]], h["cells"][h["clist"]])
        assert len(d["cells"]) == len(h["cells"])


# the leaf levels come from sliding maxima over ncrit + 1 particles, at most
# 1025 at a time, in blocks of 2048; nodes are counted in blocks of 1024
@pytest.mark.parametrize("n,ncrit", [
    (1, 1), (2, 1), (3, 2), (64, 1), (1023, 16), (1024, 1023), (1025, 1024), (1026, 1025),
    (2047, 7), (2048, 2048), (2049, 2047), (5000, 1025), (9000, 3000), (4097, 4096), (3000, 1),
])
def test_treepm_lists_at_block_and_window_edges(n, ncrit):
    import pgamd
    _, x = ics.clumpy_box(n, n + ncrit, nclump=3, sigma=0.003)
    h = pgamd.treepm_lists(x, 0.07, ncrit)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), n, 0.07, ncrit), False)


@pytest.mark.parametrize("n,ncrit,nleaf,theta", [
    (2, 1, 1, 0.5), (3, 512, 1, 0.5), (1025, 1, 1, 0.7), (2049, 1500, 1100, 0.5),
    (4096, 64, 64, 0.3), (6000, 512, 8, 0.1), (3000, 3000, 8, 0.5), (2500, 7, 2, 1.5),
])
def test_bh_lists_at_block_and_window_edges(n, ncrit, nleaf, theta):
    import pgamd
    m, x = ics.hernquist(n, n)
    x[: n // 10] = x[0]  # more coincident particles than a leaf holds
    h = pgamd.bh_lists(x, m, theta, ncrit, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, theta, ncrit, nleaf), True)


# the walk's queue: entries in chunks of 256, at most 64 a group (16384 opened
# nodes), from a pool of 5 to 40 chunks a group; beyond either the build falls
# back to the depth-first walk
@pytest.mark.parametrize("n,ncrit,nleaf,theta", [
    (2000, 2000, 1, 0.01), (20000, 20000, 1, 0.01), (60000, 60000, 1, 0.01),
    (30000, 64, 1, 0.05), (8000, 8, 3, 0.2), (700, 700, 700, 0.5), (5000, 32, 8, 40.0),
])
def test_bh_lists_at_queue_edges(n, ncrit, nleaf, theta):
    import pgamd
    m, x = ics.hernquist(n, n + 1)
    h = pgamd.bh_lists(x, m, theta, ncrit, nleaf)
    d_x, d_m = dev(x), dev(m)
    check(h, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, theta, ncrit, nleaf), True)
