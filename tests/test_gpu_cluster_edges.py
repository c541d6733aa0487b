"""Clusters at the edges of the j-tiles and of the chunks of i-particles, with
no softening (a self pair that is not left out gives NaN)."""
import numpy as np
import pytest

import ics

pytestmark = pytest.mark.gpu

BOUND = (32 + 255) * 2.0 ** -24  # roundings of an FP32 term and of a sum of 256 of them


def dev(a):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    torch.cuda.synchronize()
    return t


# tiles of 128, 256 and 512 j; chunks of 256 i, wavefronts of 64 with and
# without an i; `first` moves the chunks off the tiles
@pytest.mark.parametrize("tile", [128, 256, 512])
@pytest.mark.parametrize("first", [0, 100])
def test_clusters_at_tile_edges(tile, first):
    import torch

    import pgamd
    sizes = [2, 64, 65, 128, 129, 193, 255, 256, 257, 385, 511, 512, 513, 641, 769, 1025]
    coff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    parts = [ics.plummer(n, n) for n in sizes]
    m = np.concatenate([p[0] for p in parts])
    x = np.concatenate([p[1] + 3 * k for k, p in enumerate(parts)])
    v = np.concatenate([p[2] for p in parts])
    items = [(c, i) for c, n in enumerate(sizes)
             for i in sorted({0, *range(min(first, n - 1) if first else 0, n, 256)})]
    n = len(m)
    g6 = pgamd.G6()
    acc, jrk = (torch.full((n, 3), np.nan, dtype=torch.float64, device="cuda") for _ in range(2))
    pot = torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
    d = [dev(np.array(items, np.int32).ravel()), dev(coff), dev(x), dev(v), dev(m),
         dev(np.zeros(len(sizes), np.float32))]
    assert g6.lib.pg6_cluster_set_launch(tile, -1) == 0
    try:
        assert g6.lib.pg6_cluster_force(len(items), *[t.data_ptr() for t in d], acc.data_ptr(),
                                        jrk.data_ptr(), pot.data_ptr(), None) == 0
        torch.cuda.synchronize()
    finally:
        g6.lib.pg6_cluster_set_launch(0, 0)
    a, j, p = acc.cpu().numpy(), jrk.cpu().numpy(), pot.cpu().numpy()
    v = v.astype(np.float32).astype(np.float64)
    for lo, hi in zip(coff[:-1], coff[1:]):
        dx, dv = x[None, lo:hi] - x[lo:hi, None], v[None, lo:hi] - v[lo:hi, None]
        r2 = (dx * dx).sum(2)
        np.fill_diagonal(r2, np.inf)
        mr3 = (m[lo:hi] / (r2 * np.sqrt(r2)))[:, :, None]
        rv = ((dx * dv).sum(2) / r2)[:, :, None]
        ra = ((np.abs(dx) * np.abs(dv)).sum(2) / r2)[:, :, None]
        for got, terms, size in (
            (a[lo:hi], mr3 * dx, mr3 * np.abs(dx)),
            (j[lo:hi], mr3 * (dv - 3 * rv * dx), mr3 * (np.abs(dv) + 3 * ra * np.abs(dx))),
            (p[lo:hi], -m[lo:hi] / np.sqrt(r2), m[lo:hi] / np.sqrt(r2)),
        ):
            assert np.all(np.abs(got - terms.sum(1)) <= BOUND * size.sum(1)), (hi - lo)
