"""Meshes whose transforms along x run with the Green's function (powers of two
from 32 to 256), next to ones that take whole three-dimensional transforms."""
import numpy as np
import pytest

import pm_oracle as P
from test_gpu_pm_bricks import gpu_force

pytestmark = pytest.mark.gpu


# in an order that changes between the two kinds and comes back to a mesh
@pytest.mark.parametrize("mesh", [32, 30, 64, 66, 128, 16, 32, 256, 128])
def test_mesh_force_by_planes(mesh):
    rng = np.random.default_rng(mesh)
    n = 4000
    x = rng.random((n, 3)) ** 2
    m = rng.uniform(0.5, 1.5, n) / n
    a = 3.0 / mesh
    got, want = gpu_force(x, m, mesh, a), P.pm_force(x, m, mesh, a)
    # the bound of the mesh tests: FP64 throughout, 64-bit fixed-point density
    assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
