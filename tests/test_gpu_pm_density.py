"""The particle mesh on meshes of up to and of more than 4096 bricks, whose
particles are counted in LDS by one block or scanned in tiles of 1024 bricks, at
the density from which they are sorted, against the oracle."""
import numpy as np
import pytest

import pm_oracle as P
from test_gpu_pm_bricks import gpu_force

pytestmark = pytest.mark.gpu


# 4096 bricks at 128, 4913 at 130 and 136 (5 tiles), 6859 at 152, 15625 at 200: sorted
# from 3 a brick
@pytest.mark.parametrize("n,mesh", [
    (12287, 128), (12288, 128), (14738, 130), (14739, 130), (60000, 136), (21000, 152), (46874, 200),
    (46875, 200),
])
def test_mesh_force_at_the_sorting_density(n, mesh):
    rng = np.random.default_rng(n + mesh)
    x = rng.random((n, 3))
    m = rng.uniform(0.5, 1.5, n) / n
    got, want = gpu_force(x, m, mesh, 3.0 / mesh), P.pm_force(x, m, mesh, 3.0 / mesh)
    # the mesh tests' bound: FP64 throughout, 64-bit fixed-point density
    assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
