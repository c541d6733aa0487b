"""TreePM neighbour lists of particles at the cut-off from their groups to
within a few units in the last place, and of particles outside the box, array
for array against the host builder."""
import numpy as np
import pytest

import ics
from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu


# distances rcut (1 + k 2^-52), k = -4 .. 4, along an axis and across; jitters
# of the size of FP32 roundings
@pytest.mark.parametrize("cells,jitter", [(8, 0.0), (16, 2e-16), (16, 3e-8), (13, 1e-6), (5, 1e-7)])
def test_lists_at_the_cutoff(cells, jitter):
    import pgamd
    rng = np.random.default_rng(cells)
    rcut = 1.0 / cells
    g = np.stack(np.meshgrid(*[np.arange(cells)] * 3, indexing="ij"), -1).reshape(-1, 3) * rcut
    x = np.concatenate([g, g * (1 + rng.integers(-4, 5, g.shape) * 2.0 ** -52)])
    x = (x + jitter * rng.uniform(-1, 1, x.shape)) % 1.0
    h = pgamd.treepm_lists(x, rcut, 2)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), len(x), rcut, 2), False)


@pytest.mark.parametrize("span", [1.0, 3.0, 40.0])
def test_lists_outside_the_box(span):
    import pgamd
    _, x = ics.clumpy_box(3000, 5, nclump=3, sigma=0.01)
    x[::7] = span * (2 * x[::7] - 1)
    h = pgamd.treepm_lists(x, 0.07, 16)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), len(x), 0.07, 16), False)
