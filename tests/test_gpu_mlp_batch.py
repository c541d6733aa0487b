"""The learned cut-off's batch kernel at the sizes where its slices, units and
queues end: pair sums against the network in FP64 (oracle/mlp_oracle.py)."""
import numpy as np
import pytest

import mlp_oracle as M

pytestmark = pytest.mark.gpu

RC, R0 = 3.0 / 64, 0.1 / 64


@pytest.fixture(scope="module")
def tab():
    import pgamd
    t = pgamd.G5Table()
    t.lib.pg5_gen_s2_force_table(R0, RC)
    return t


def network(seed):
    rng = np.random.default_rng(seed)
    p = np.zeros(M.NP)
    p[:16], p[16:32] = 4 * rng.uniform(-1, 1, 16), 2 * rng.uniform(-1, 1, 16)
    p[32:288], p[288:304] = 0.43 * rng.uniform(-1, 1, 256), 0.5 * rng.uniform(-1, 1, 16)
    p[304:] = rng.uniform(-1, 1, 17)
    return p


def expected(xi, xj, m, p, form):
    """acc and its error bound.  A pair's terms (Newtonian and network) carry a
    relative rounding error of at most 3e-5 of their sizes (FP32 network: 16
    products of size up to 20 in the exponent of an activation; FP32 sums of up
    to 256 pairs), and the separations, FP32 offsets from the group's first
    particle, one of 2^-23 of the box over r per power of r (4 of them)."""
    d = xj[None] - xi[:, None]
    r = np.sqrt((d * d).sum(-1))
    size = np.abs(2 * p[304:320]).sum() + abs(p[320] - p[304:320].sum())
    ok = (r > 0) & (r < RC)
    s = np.where(ok, r, RC)
    if form == 1:
        near = s < R0
        u = M.forward(p, (s / RC).ravel()).reshape(s.shape)
        c = M.forward(p, np.minimum(s / R0, 1).ravel()).reshape(s.shape)
        f = np.where(near, c / R0 ** 3, 1 / s ** 3) - u / RC ** 3
        a = np.where(near, size / R0 ** 3, 1 / s ** 3) + size / RC ** 3
    else:
        y = M.forward(p, np.sqrt(s / RC).ravel()).reshape(s.shape)
        f, a = y / (s ** 3 + R0 ** 3), size / (s ** 3 + R0 ** 3)
    f, a = np.where(ok, f, 0.0), np.where(ok, a, 0.0)
    box = np.abs(np.concatenate([xi, xj]) - xi[0]).max()
    tol = (a * m * r * (3e-5 + 4 * 2.0 ** -23 * box / s)).sum(1)
    return ((f * m)[..., None] * d).sum(1), tol


@pytest.mark.parametrize("form", [1, 0])
@pytest.mark.parametrize("sizes", [
    [(1, 1), (1, 64), (16, 65), (17, 255)],
    [(32, 257), (33, 63), (64, 256), (63, 300)],
    [(65, 129), (128, 511), (127, 512)],
    [(129, 64), (192, 257), (193, 700), (256, 256), (255, 1)],
    [(257, 130), (400, 513), (700, 90)],
])
def test_learned_batch_matches_oracle_at_its_edges(tab, sizes, form):
    import torch
    p = network(3 + form)
    tab.mlp_set_params(p, form, RC, R0)
    rng = np.random.default_rng(sum(a * 7 + b for a, b in sizes))
    x, m, ioff, icnt, ilist, joff, jcnt, jlist = [], [], [], [], [], [], [], []
    n = 0
    for ni, nj in sizes:
        q = max(ni, nj)
        c = 0.5 + RC * rng.uniform(-1, 1, (q, 3))  # about half the pairs in reach
        if q > 3:  # pairs inside the S2 core, and one i-particle's own twin
            c[1::4] = c[0::4][: len(c[1::4])] + 0.4 * R0 * rng.uniform(-1, 1, (len(c[1::4]), 3))
            c[3] = c[2]
        x.append(c)
        m.append(rng.uniform(0.5, 1.5, q))
        ioff.append(len(ilist)), icnt.append(ni), ilist.extend(n + rng.permutation(q)[:ni])
        joff.append(len(jlist)), jcnt.append(nj), jlist.extend(n + rng.permutation(q)[:nj])
        n += q
    x, m = np.concatenate(x), np.concatenate(m)
    _, xs = tab.table()
    pos4 = np.concatenate([x.astype(np.float32) * np.float32(xs), m[:, None]], 1).astype(np.float32)
    dev = lambda a, t: torch.from_numpy(np.ascontiguousarray(a, t)).cuda()  # noqa: E731
    order = np.argsort(-np.array(icnt) * np.array(jcnt))
    idx = [dev(a, np.int32) for a in (ioff, icnt, ilist, joff, jcnt, jlist, order)]
    d_pos, d_x = dev(pos4, np.float32), dev(x, np.float64)
    acc = torch.full((n, 3), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert tab.lib.pg5t_batch_force(0, len(sizes), *[t.data_ptr() for t in idx], d_pos.data_ptr(),
                                    d_x.data_ptr(), acc.data_ptr(), 1, None) == 0
    torch.cuda.synchronize()
    acc = acc.cpu().numpy()
    listed = np.zeros(n, bool)
    m32 = m.astype(np.float32).astype(np.float64)
    for g, (ni, nj) in enumerate(sizes):
        i = np.array(ilist[ioff[g]:ioff[g] + ni])
        j = np.array(jlist[joff[g]:joff[g] + nj])
        listed[i] = True
        a, tol = expected(x[i], x[j], m32[j], p, form)
        err = np.linalg.norm(acc[i] - a, axis=1)
        assert np.all(err <= tol), (ni, nj, float((err / np.maximum(tol, 1e-300)).max()))
    assert np.all(acc[~listed] == 7.0)
