"""Block steps over the force splits: one to three ranges per lane and wavefront
per particle, up to 16 ranges and four lanes per particle, short and long
ranges; every active particle against the restated integrator."""
import numpy as np
import pytest

import ics
import oracle as O

pytestmark = pytest.mark.gpu

ETA_S, ETA, DTMAX, EPS2 = 0.01, 0.2, 0.125, (1 / 128) ** 2


@pytest.fixture(scope="module")
def g6():
    import pgamd
    g = pgamd.G6()
    yield g
    g.lib.pg6_hermite_end()


def check_force(i, x, v, xj, vj, m, s):
    """Force, jerk and potential of particle i against FP64 sums.  The terms
    are FP32: each goes through at most 32 roundings of 2^-24 (the square
    root's reciprocal, good to one unit, enters cubed), and a sum of up to 256
    terms through 255 more; all relative to the sum of the terms' sizes."""
    dx, dv = np.delete(xj - x, i, 0), np.delete(vj - v, i, 0)
    mj = np.delete(m, i)
    r2 = (dx * dx).sum(1) + EPS2
    rv = (dx * dv).sum(1) / r2
    mr3 = mj / (r2 * np.sqrt(r2))
    bound = (32 + 255) * 2.0 ** -24
    for got, terms, size in (
        (s["a"][i], mr3[:, None] * dx, mr3[:, None] * np.abs(dx)),
        (s["j"][i], mr3[:, None] * (dv - 3 * rv[:, None] * dx),
         mr3[:, None] * (np.abs(dv) + 3 * ((np.abs(dx) * np.abs(dv)).sum(1) / r2)[:, None]
                         * np.abs(dx))),
        (s["pot"][i], -mj / np.sqrt(r2), mj / np.sqrt(r2)),
    ):
        assert np.all(np.abs(got - terms.sum(0)) <= bound * size.sum(0)), i


# ranges of 128 addresses up to 16 (quads) and from 17 on (wavefronts), of 256
# beyond 2^14 particles, 65 and 129 of them (a second and third one a lane); of
# 512 from 65536 on; to the window's end, where all particles move
@pytest.mark.parametrize("n,steps", [
    (63, 0), (65, 0), (1025, 0), (2048, 0), (2049, 0), (2176, 0), (4400, 0), (16384, 3),
    (16700, 3), (33000, 3), (70001, 2),
])
def test_steps_over_the_splits(g6, n, steps):
    m, x, v = ics.plummer(n, n)
    g6.hermite_init(x, v, m, EPS2, ETA_S, ETA, DTMAX)
    idx = np.arange(n, dtype=np.int32)
    if not steps:  # one step short of the window's end, then that one and two more
        s0 = g6.hermite_state()
        g6.hermite_run(DTMAX - 1e-9 - s0["dt"].min())
        steps = 3
    s0 = g6.hermite_state()
    for step in range(steps):
        tn = (s0["t"] + s0["dt"]).min()
        act = s0["t"] + s0["dt"] == tn
        _, nact = g6.hermite_step()
        s1 = g6.hermite_state()
        assert nact == act.sum(), step
        xp, vp = O.hermite_predict(tn, s0["t"][act], s0["x"][act], s0["v"][act], s0["a"][act],
                                   s0["j"][act])
        x1, v1, dtn = O.hermite_correct(ETA, DTMAX, s0["t"][act], s0["dt"][act], s0["a"][act],
                                        s0["j"][act], xp, vp, s1["a"][act], s1["j"][act])
        np.testing.assert_array_equal(s1["x"][act], x1)
        np.testing.assert_array_equal(s1["v"][act], v1)
        np.testing.assert_array_equal(s1["dt"][act], dtn)
        np.testing.assert_array_equal(s1["t"][act], 0.0 if tn == DTMAX else tn)
        xj, vj = O.pg6_predict(tn, s0["x"], s0["v"], s0["a"] / 2, s0["j"] * (1.0 / 6.0), s0["t"])
        vj = vj.astype(np.float32).astype(np.float64)
        for k, i in list(enumerate(np.flatnonzero(act)))[:64]:
            check_force(i, xp[k], vp[k].astype(np.float32).astype(np.float64), xj, vj, m, s1)
        for k in ("x", "v", "a", "j", "dt"):
            np.testing.assert_array_equal(s1[k][~act], s0[k][~act], err_msg=k)
        s0 = s1
