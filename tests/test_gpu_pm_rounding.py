"""The particle mesh where the rounding of x M decides between two mesh points:
positions within a few units in the last place of the halfway points, inside and
outside the box, in the sorted and in the direct path."""
import numpy as np
import pytest

import pm_oracle as P
from test_gpu_pm_bricks import gpu_force

pytestmark = pytest.mark.gpu


# sorted from 3 particles per brick of 8^3 points: (mesh / 8)^3 bricks, rounded up
@pytest.mark.parametrize("n,mesh", [
    (1000, 10), (1000, 12), (3000, 20), (4000, 22), (4000, 26), (9000, 40), (9000, 100),
    (20, 10), (60, 20), (500, 100),
])
def test_mesh_force_at_halfway_points(n, mesh):
    rng = np.random.default_rng(n + mesh)
    k = rng.integers(-mesh, 2 * mesh, (n, 3))
    k[:: 3] = -1  # x = -0.5 / mesh, where fma(x, mesh, 0.5) and x * mesh + 0.5 differ
    x = (k + 0.5) / mesh
    ulps = rng.integers(-2, 3, x.shape)
    ulps[:: 6] = 0
    x = x + ulps * np.spacing(x)
    some = rng.random(x.shape) < 0.2
    x = np.where(some, rng.random(x.shape), x)
    m = rng.uniform(0.5, 1.5, n) / n
    a = 3.0 / mesh
    got, want = gpu_force(x, m, mesh, a), P.pm_force(x, m, mesh, a)
    # the mesh tests' bound: FP64 throughout, 64-bit fixed-point density (the two
    # points' stencils agree at the halfway point, so either one is right)
    assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
