"""A Barnes-Hut build with little device memory left: the opening pool is given
up for the depth-first walk, which needs none, instead of ending the program."""
import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def test_bh_lists_without_memory_for_the_pool():
    import pgamd
    import torch
    n, theta, ncrit = 1 << 17, 0.3, 16
    m, x = ics.hernquist(n, 21)
    h = pgamd.bh_lists(x, m, theta, ncrit, 8)
    d_x, d_m = dev(x), dev(m)
    taken, block = [], 16 * GIB
    try:
        # leave 3 GiB: the lists take 1.3, the pool would take 2.3
        while (spare := torch.cuda.mem_get_info()[0] - 3 * GIB) >= GIB // 64 and block > GIB // 64:
            try:
                taken.append(torch.empty(min(spare, block), dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:  # what is left is in smaller pieces
                block //= 2
        L = pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), n, theta, ncrit, 8)
    finally:
        taken.clear()
        torch.cuda.empty_cache()
    check(h, L, False)
