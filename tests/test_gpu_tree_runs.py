"""The list builds' sort where many particles share the upper bits of their keys:
runs of up to 512 are put in order by counting, longer ones by a sort of all
bits; array for array against the host builder."""
import numpy as np
import pytest

from test_gpu_tree_edges import check, dev

pytestmark = pytest.mark.gpu


# 2^18 particles and more are sorted by counting: first the upper 40 bits of
# the keys (cells of 2^-13 of the box an axis; 2^-14 along x)
@pytest.mark.parametrize("run", [511, 512, 513, 700, 1023, 1024, 1025, 40000])
@pytest.mark.parametrize("n,every", [(262144, False), (263001, True)])
def test_lists_of_particles_with_equal_upper_bits(n, every, run):
    import pgamd
    rng = np.random.default_rng(run)
    x = rng.random((n, 3))
    cells = n // (8 * run) + 1 if every else 1  # an eighth of the particles, or one run
    for c in range(cells):
        corner = rng.integers(1, 8191, 3) / 8192
        x[c * run:(c + 1) * run] = corner + (rng.integers(0, 128, (run, 3)) + 0.5) / 2 ** 21
    x = np.ascontiguousarray(rng.permutation(x))
    h = pgamd.treepm_lists(x, 0.02, 64)
    d_x = dev(x)
    check(h, pgamd.DevLists.treepm(d_x.data_ptr(), n, 0.02, 64), False)
