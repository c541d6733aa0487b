"""The particle mesh at the edges of its brick sort: meshes that bricks of 8
points do not divide, chunk and density limits, positions outside the box."""
import numpy as np
import pytest

import pm_oracle as P

pytestmark = pytest.mark.gpu


def gpu_force(x, m, mesh, a):
    import pgamd
    import torch
    T = pgamd.G5Table()
    d_x, d_m = torch.from_numpy(np.ascontiguousarray(x)).cuda(), torch.from_numpy(m).cuda()
    acc = torch.empty((len(m), 3), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert T.lib.pg5t_pm_force(len(m), d_x.data_ptr(), d_m.data_ptr(), mesh, a, acc.data_ptr(),
                               None) == 0
    torch.cuda.synchronize()
    return acc.cpu().numpy()


# bricks: mesh 8 -> 1, 10, 12, 14 and 16 -> 8, 18 -> 27, 32 -> 64, 136 -> 4913
# (more than are counted in LDS); sorted from 3 particles per brick
@pytest.mark.parametrize("n,mesh,where", [
    (1, 8, "box"), (2, 8, "box"), (3, 8, "box"), (23, 10, "box"), (24, 10, "box"),
    (80, 18, "box"), (81, 18, "box"), (511, 16, "cell"), (512, 16, "cell"), (513, 16, "cell"),
    (1025, 32, "cell"), (4097, 32, "corner"), (5000, 12, "corner"), (3000, 14, "outside"),
    (191, 32, "outside"), (14738, 136, "box"), (14739, 136, "corner"),
])
def test_mesh_force_at_brick_edges(n, mesh, where):
    rng = np.random.default_rng(n + mesh)
    x = rng.random((n, 3))
    if where == "cell":  # every particle near one mesh point
        x = (5 + 0.4 * (x - 0.5)) / mesh
    elif where == "corner":  # around the periodic corner and the last brick's end
        x = np.where(rng.random((n, 1)) < 0.5, (2 * x - 1) / mesh % 1.0, x)
    elif where == "outside":
        x = 3 * x - 1
        x[:3] = [[1.0, 0.0, 1.0], [-1.0, 2.0, 1.5 / mesh], [1.0 - 0.5 / mesh] * 3]
    m = rng.uniform(0.5, 1.5, n) / n
    a = 3.0 / mesh
    got, want = gpu_force(x, m, mesh, a), P.pm_force(x, m, mesh, a)
    # the bound of the mesh tests: FP64 throughout, 64-bit fixed-point density
    scale = np.abs(want).max()
    if n > 1:
        assert np.abs(got - want).max() <= 1e-9 * scale
    else:  # a particle's own mesh force vanishes but for rounding
        assert np.abs(got).max() <= 1e-9 * mesh ** 2
