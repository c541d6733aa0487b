"""Performance cases of the pairwise-gravity libraries: what N-body programs
call, through the public entry points (the Python mirror ``pgamd`` of the C
ABI), with sizes taken from the benchmark configurations and the tests.

``listed()`` are the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` makes what a program has in hand before the call,
``run(state)`` is one pass, ``work(case)`` the bytes and flops a pass cannot do
without, ``exact(case, seed)`` the outputs in 64 bits from plain numpy / torch.

Flops follow the reference's conventions: 38 per softened pair force, 60 per
force + jerk pair, 71 per quadrupole cell.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "phantom-grape_amd"))

import ics  # noqa: E402
import pgamd  # noqa: E402


def listed():
    return [
        # One leapfrog step of a small N-body program on the GRAPE-5 host API:
        # load the j-particles, force on all of them (the reference's `direct`
        # benchmark has 4096 particles and this softening).
        dict(name="g5_host_4096", kind="g5_host", n=4096, eps=0.02),
        # The same step with the particles already on the GPU, at the direct-sum
        # benchmark's size.
        dict(name="g5_dev_16384", kind="g5_dev", ni=16384, nj=16384, eps=1 / 64, sym=False),
        # One call of a block-time-step integrator on the GRAPE-6 host API: 48
        # i-particles (the board's pipelines) against all j, neighbour included.
        dict(name="g6_host_48", kind="g6_host", ni=48, nj=16384, eps=1 / 256),
        # A block step with the i-particles on the GPU: every particle of the
        # headline configuration moves (start-up passes and window ends).
        dict(name="g6_dev_65536", kind="g6_dev", ni=65536, nj=65536, eps=1 / 256, nn=True),
        # A whole integration on the GPU: the reference's published GRAPE-6
        # benchmark setup, from initial conditions to the state at t = 1/8.
        dict(name="hermite_16384", kind="hermite", n=16384, t=1 / 8),
        # Many independent star clusters of uneven size, one force pass each.
        dict(name="clusters_4096", kind="clusters", ncl=4096, nmin=64, nmax=4096),
        # The parts of one TreePM force step of a clumpy box, positions on the
        # GPU: interaction lists, short range by the table, long range on the
        # mesh; and the short range by the learned cut-off on a smaller box.
        dict(name="treepm_lists_2p20", kind="treepm_lists", n=1 << 20),
        dict(name="treepm_table_2p20", kind="treepm_table", n=1 << 20, frc=6, order=1,
             origin=False),
        dict(name="treepm_mlp_2p18", kind="treepm_mlp", n=1 << 18, origin=True),
        dict(name="pm_mesh_2p20", kind="pm", n=1 << 20, mesh=128),
        # The two parts of a Barnes-Hut force step of a halo: particle and
        # quadrupole-cell lists, and the force over them.
        dict(name="bh_lists_2p21", kind="bh_lists", n=1 << 21, theta=0.5),
        dict(name="bh_force_2p21", kind="bh_force", n=1 << 21, theta=0.5, eps=1 / 128),
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm, mostly odd
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["g5_host", "g5_dev", "g6_host", "g6_dev", "hermite", "clusters",
                       "treepm_lists", "treepm_table", "treepm_mlp", "pm", "bh_lists",
                       "bh_force"])
    if kind == "g5_host":
        return dict(kind=kind, n=size(256, 16384), eps=rng.choice([0.02, 1 / 64, 1 / 256]))
    if kind == "g5_dev":
        return dict(kind=kind, ni=size(64, 65536), nj=size(1024, 131072),
                    eps=rng.choice([1 / 64, 1 / 128]), sym=rng.random() < 0.3)
    if kind == "g6_host":
        return dict(kind=kind, ni=size(1, 256), nj=size(1024, 65536), eps=1 / 256)
    if kind == "g6_dev":
        nj = size(1024, 65536)
        return dict(kind=kind, ni=min(nj, size(32, 65536)), nj=nj, eps=1 / 256,
                    nn=rng.random() < 0.7)
    if kind == "hermite":
        return dict(kind=kind, n=size(512, 16384), t=rng.choice([1 / 64, 1 / 32, 1 / 16]))
    if kind == "clusters":
        nmin = size(16, 256)
        return dict(kind=kind, ncl=size(64, 4096), nmin=nmin, nmax=size(nmin + 64, 4096))
    if kind == "treepm_lists":
        return dict(kind=kind, n=size(1 << 14, 1 << 20))
    if kind == "treepm_table":
        return dict(kind=kind, n=size(1 << 14, 1 << 20), frc=rng.choice([5, 6]),
                    order=rng.choice([1, 2]), origin=rng.random() < 0.5)
    if kind == "treepm_mlp":
        return dict(kind=kind, n=size(1 << 13, 1 << 18), origin=rng.random() < 0.5)
    if kind == "pm":
        return dict(kind=kind, n=size(1 << 14, 1 << 20), mesh=2 * size(16, 64))
    return dict(kind=kind, n=size(1 << 14, 1 << 21), theta=rng.choice([0.5, 0.6, 0.75]),
                **(dict(eps=1 / 128) if kind == "bh_force" else {}))


# ------------------------------------------------------------------ handles
@functools.lru_cache(None)
def g5(sym):
    return pgamd.G5(symmetric=sym)


@functools.lru_cache(None)
def g6():
    return pgamd.G6()


@functools.lru_cache(None)
def g5t():
    return pgamd.G5Table()


@functools.lru_cache(None)
def stream():
    # torch's default stream has the null handle, which the libraries read as
    # their own stream: a program that mixes the two gives them one of its own
    return torch.cuda.Stream().cuda_stream


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def empty(*shape, dtype=torch.float64):
    return torch.empty(shape, dtype=dtype, device="cuda")


class DevArray:
    """A device array of a list handle, as torch reads it (no copy); keeps the
    handle alive."""

    def __init__(self, lists, name, shape, typestr):
        self.lists = lists
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, strides=None, version=2,
                                             data=(lists.ptr(name), False))


def list_tensors(DL, names):
    i = DL.info()
    size = dict(pos=(i["np"], 3), src=(i["np"],), ilist=(i["ni"],), jlist=(i["nj"],),
                clist=(i["nc"],), cells=(i["ncells"], 10))
    return {k: torch.as_tensor(DevArray(DL, k, size.get(k, (i["ngroups"],)),
                                        "<f8" if k in ("pos", "cells") else "<i4"), device="cuda")
            for k in names}


# ------------------------------------------------------------------ inputs
GROUP = ("ioff", "icnt", "ilist", "joff", "jcnt", "jlist", "order")
CELLS = ("ioff", "icnt", "ilist", "joff", "jcnt", "jlist", "coff", "ccnt", "clist", "order")


def mesh_of(n):
    """Mesh of a TreePM box of n particles: 128 at 2^20, as many particles per
    mesh cell elsewhere."""
    return 2 * round(64 * (n / 2 ** 20) ** (1 / 3))


def split_of(n):
    """(eps_PP, eps_PM): the S2 split of that mesh, eps_PM is the cut-off."""
    return 0.1 / mesh_of(n), 3.0 / mesh_of(n)


def set_table(n, frc, order):
    L = g5t().lib
    L.pg5_set_table_order(1)
    L.pg5_gen_s2_force_table(*split_of(n))
    assert L.pg5_set_table_frc_bit(frc) == 0 and L.pg5_set_table_order(order) == 0


@functools.lru_cache(None)
def network():
    """Parameters of a 1-16-16-1 tanh network of the S2 unit shape: seeded
    hidden layers, the output layer by regularised least squares."""
    rng = np.random.default_rng(16)
    p = np.zeros(321)
    p[:16], p[16:32] = 4 * rng.uniform(-1, 1, 16), 2 * rng.uniform(-1, 1, 16)
    p[32:288], p[288:304] = rng.uniform(-1, 1, 256), 0.5 * rng.uniform(-1, 1, 16)
    u = np.linspace(0, 1, 4097)
    h = np.tanh((2 * u[:, None] - 1) * p[:16] + p[16:32])
    h = np.tanh(h @ p[32:288].reshape(16, 16).T + p[288:304])
    A = np.concatenate([h, np.ones((len(u), 1))], 1)
    p[304:] = np.linalg.solve(A.T @ A + 1e-4 * np.eye(17), A.T @ s2(u, 1.0))
    return p


@functools.lru_cache(4)
def model(nj):
    """The j-particles of a GRAPE-6 board: a Plummer sphere with the sphere's
    mean acceleration and jerk, each last updated one block step before t = 1."""
    m, x, v = ics.plummer(nj, 65536)
    b = 3 * np.pi / 16
    s = (x * x).sum(1, keepdims=True) + b * b
    a = -x / s ** 1.5
    j = -v / s ** 1.5 + 3 * x * (x * v).sum(1, keepdims=True) / s ** 2.5
    dt = 0.02 * np.linalg.norm(a, axis=1) / np.linalg.norm(j, axis=1)
    dt = 2.0 ** -np.clip(np.ceil(-np.log2(dt)), 3, 12)
    return m, x, v, a / 2, j / 6, 1.0 - dt


def predicted(nj, t):
    m, x, v, a2, j6, tj = model(nj)
    h = (t - tj)[:, None]
    return x + v * h + a2 * h * h + j6 * h ** 3, v + 2 * a2 * h + 3 * j6 * h * h


def block(case, seed):
    """A block of a block step: its time, and the i-particles at that time."""
    rng = np.random.default_rng(seed)
    t = 1.0 - 2.0 ** -12 * rng.random()
    sel = np.sort(rng.choice(case["nj"], case["ni"], replace=False))
    x, v = predicted(case["nj"], t)
    return t, x[sel], v[sel], sel.astype(np.int32)


def halves(case, seed):
    """i- and j-particles of a direct sum: an i-set taken from the j-set, or
    probes drawn from the same sphere where it is larger."""
    m, x, _ = ics.plummer(case["nj"], seed)
    rng = np.random.default_rng(seed + 1)
    if case["ni"] <= case["nj"]:
        xi = x[np.sort(rng.choice(case["nj"], case["ni"], replace=False))]
    else:
        xi = ics.plummer(case["ni"], seed + 2)[1]
    e2i = np.full(case["ni"], case["eps"] ** 2)
    e2j = (case["eps"] * rng.uniform(0.5, 1.5, case["nj"])) ** 2 if case["sym"] else None
    f4 = lambda p, w: np.concatenate([p, w[:, None]], 1).astype(np.float32)  # noqa: E731
    return f4(xi, e2i), f4(x, m), None if e2j is None else e2j.astype(np.float32)


def star_clusters(case, seed):
    """Plummer spheres of log-uniform sizes (the case's own), one after the other."""
    size = ics.cluster_sizes(case["ncl"], case["ncl"], case["nmin"], case["nmax"])
    coff = np.concatenate([[0], np.cumsum(size)]).astype(np.int32)
    n, rng = int(coff[-1]), np.random.default_rng(seed)

    def directions():
        d = rng.normal(size=(n, 3))
        return d / np.linalg.norm(d, axis=1, keepdims=True)

    r = 1 / np.sqrt(((1 + 1 / 400) ** -1.5 * (1 - rng.random(n))) ** (-2 / 3) - 1)
    speed = np.sqrt(rng.beta(1.5, 4.5, n)) * np.sqrt(2) * (1 + r * r) ** -0.25
    b = 3 * np.pi / 16
    x, v = directions() * (b * r)[:, None], directions() * (speed / np.sqrt(b))[:, None]
    return size, coff, x, v, np.repeat(1.0 / size, size), ((4.0 / size) ** 2).astype(np.float32)


def turned(x, seed):
    """The same body of particles in another orientation and input order: how
    many groups and list entries it has depends on neither, so that passes on
    other inputs return arrays of the same lengths."""
    rng = np.random.default_rng(seed)
    return np.ascontiguousarray(x[rng.permutation(len(x))][:, rng.permutation(3)])


def treepm_lists_of(n, seed):
    m, x = ics.clumpy_box(n, seed)
    d_x, d_m = dev(x), dev(m)
    torch.cuda.synchronize()
    return m, d_m, pgamd.DevLists.treepm(d_x.data_ptr(), n, split_of(n)[1], 256, stream=stream())


def bh_lists_of(case, seed):
    m, x = ics.hernquist(case["n"], seed)
    d_x, d_m = dev(x), dev(m)
    torch.cuda.synchronize()
    return m, d_m, pgamd.DevLists.bh(d_x.data_ptr(), d_m.data_ptr(), case["n"], case["theta"], 512,
                                     8, stream=stream())


def prepare(case, seed):
    k, s = case["kind"], dict(case=case)
    if k == "g5_host":
        s["m"], s["x"], _ = ics.plummer(case["n"], seed)
        g5(False)
    elif k == "g5_dev":
        xi, xj, e2j = halves(case, seed)
        s.update(xi=dev(xi), xj=dev(xj), e2j=None if e2j is None else dev(e2j),
                 acc=empty(case["ni"], 3), pot=empty(case["ni"]))
        g5(case["sym"])
    elif k in ("g6_host", "g6_dev"):
        m, x, v, a2, j6, tj = model(case["nj"])
        assert g6().set_j_bulk(x, v, a2, j6, m, tj, np.arange(case["nj"])) == 0
        s["t"], s["x"], s["v"], s["id"] = block(case, seed)
        if k == "g6_dev":
            ni = case["ni"]
            s.update(x=dev(s["x"]), v=dev(s["v"]), id=dev(s["id"]), acc=empty(ni, 3),
                     jrk=empty(ni, 3), pot=empty(ni))
            if case["nn"]:
                s.update(nnb=empty(ni, dtype=torch.int32), rnnb=empty(ni, dtype=torch.float32))
    elif k == "hermite":
        s["m"], s["x"], s["v"] = ics.plummer(case["n"], seed)
        g6()
    elif k == "clusters":
        _, coff, x, v, m, e2 = star_clusters(case, seed)
        s.update(items=dev(g6().cluster_items(coff)), coff=dev(coff), x=dev(x), v=dev(v), m=dev(m),
                 e2=dev(e2), acc=empty(len(m), 3), jrk=empty(len(m), 3), pot=empty(len(m)))
    elif k == "treepm_lists":
        s["x"] = dev(turned(ics.clumpy_box(case["n"], 20)[1], seed))
    elif k in ("treepm_table", "treepm_mlp"):
        set_table(case["n"], case.get("frc", 6), case.get("order", 1))
        if k == "treepm_mlp":
            pp, pm = split_of(case["n"])
            g5t().mlp_set_params(network(), 1, pm, pp)
        _, d_m, DL = treepm_lists_of(case["n"], seed)
        np_ = DL.info()["np"]
        s.update(lists=DL, ng=DL.info()["ngroups"], pos=empty(np_, 4, dtype=torch.float32),
                 acc=torch.zeros((np_, 3), dtype=torch.float64, device="cuda"))
        DL.pack(d_m.data_ptr(), g5t().table()[1], s["pos"].data_ptr(), None, stream())
        torch.cuda.synchronize()
    elif k == "pm":
        m, x = ics.clumpy_box(case["n"], seed)
        s.update(x=dev(x), m=dev(m), acc=empty(case["n"], 3))
        g5t()
    elif k == "bh_lists":
        m, x = ics.hernquist(case["n"], 21)
        s.update(x=dev(turned(x, seed)), m=dev(m))
    else:
        _, d_m, DL = bh_lists_of(case, seed)
        i = DL.info()
        s.update(lists=DL, ng=i["ngroups"], pos=empty(i["np"], 4, dtype=torch.float32),
                 cells=empty(i["ncells"], 12, dtype=torch.float32), acc=empty(case["n"], 3),
                 pot=empty(case["n"]))
        DL.pack(d_m.data_ptr(), 1.0, s["pos"].data_ptr(), s["cells"].data_ptr(), stream())
        torch.cuda.synchronize()
        g5(False)
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["case"]
    k = c["kind"]
    p = lambda name: s[name].data_ptr() if s.get(name) is not None else None  # noqa: E731
    if k == "g5_host":
        G = g5(False)
        G.set_eps_to_all(c["eps"])
        G.set_xmj(0, s["x"], s["m"])
        G.set_n(c["n"])
        return G.calculate_force_on_x(s["x"])
    if k == "g5_dev":
        assert g5(c["sym"]).lib.pg5_dev_force(0, c["ni"], p("xi"), c["nj"], p("xj"), p("e2j"),
                                              p("acc"), p("pot"), stream()) == 0
        return s["acc"], s["pot"]
    if k == "g6_host":
        g6().set_ti(s["t"])
        r = g6().calc(c["nj"], s["x"], s["v"], s["id"], c["eps"] ** 2, variant="2p")
        return {q: r[q] for q in ("acc", "jrk", "pot", "nnb", "rnnb")}
    if k == "g6_dev":
        L = g6().lib
        assert L.pg6_dev_predict(c["nj"], s["t"], stream()) == 0
        assert L.pg6_dev_force(c["nj"], c["ni"], p("x"), p("v"), p("id"), c["eps"] ** 2, p("acc"),
                               p("jrk"), p("pot"), p("nnb"), p("rnnb"), stream()) == 0
        return {q: s[q] for q in ("acc", "jrk", "pot", "nnb", "rnnb") if q in s}
    if k == "hermite":
        g6().hermite_init(s["x"], s["v"], s["m"], 0.0, 0.01, 0.2, 0.125)
        g6().hermite_run(c["t"])
        return g6().hermite_state()
    if k == "clusters":
        assert g6().lib.pg6_cluster_force(s["items"].numel() // 2, p("items"), p("coff"), p("x"),
                                          p("v"), p("m"), p("e2"), p("acc"), p("jrk"), p("pot"),
                                          stream()) == 0
        return s["acc"], s["jrk"], s["pot"]
    if k == "treepm_lists":
        DL = pgamd.DevLists.treepm(p("x"), c["n"], split_of(c["n"])[1], 256, stream=stream())
        return list_tensors(DL, ("pos", "src", *GROUP))
    if k in ("treepm_table", "treepm_mlp"):
        DL = s["lists"]
        assert g5t().lib.pg5t_batch_force(0, s["ng"], *[DL.ptr(q) for q in GROUP], p("pos"),
                                          DL.ptr("pos") if c["origin"] else None, p("acc"),
                                          int(k == "treepm_mlp"), stream()) == 0
        return s["acc"][: c["n"]]
    if k == "pm":
        assert g5t().lib.pg5t_pm_force(c["n"], p("x"), p("m"), c["mesh"], 3.0 / c["mesh"], p("acc"),
                                       stream()) == 0
        return s["acc"]
    if k == "bh_lists":
        DL = pgamd.DevLists.bh(p("x"), p("m"), c["n"], c["theta"], 512, 8, stream=stream())
        return list_tensors(DL, ("pos", "src", "cells", *CELLS))
    DL = s["lists"]
    assert g5(False).lib.pg5_bh_batch(0, s["ng"], *[DL.ptr(q) for q in CELLS], p("pos"), p("cells"),
                                      c["eps"] ** 2, p("acc"), p("pot"), stream()) == 0
    return s["acc"], s["pot"]


# ------------------------------------------------------------------ work
def treepm_pairs(n):
    """Pairs within the cut-off of the clumpy box: uniform half with everyone,
    and inside each of the 64 Gaussian clumps (separations of width sqrt(2)
    sigma, sigma = 0.01)."""
    rc = split_of(n)[1]
    q = rc / (0.01 * math.sqrt(2))
    near = math.erf(q / math.sqrt(2)) - math.sqrt(2 / math.pi) * q * math.exp(-q * q / 2)
    return 0.75 * n * n * 4 / 3 * math.pi * rc ** 3 + (n / 2) ** 2 / 64 * near


def work(case):
    k = case["kind"]
    if k == "g5_host":
        return dict(bytes=64.0 * case["n"], flops=38.0 * case["n"] ** 2)
    if k == "g5_dev":
        return dict(bytes=48.0 * case["ni"] + (20.0 if case["sym"] else 16.0) * case["nj"],
                    flops=38.0 * case["ni"] * case["nj"])
    if k in ("g6_host", "g6_dev"):
        return dict(bytes=116.0 * case["nj"] + 116.0 * case["ni"],
                    flops=60.0 * case["ni"] * (case["nj"] - 1))
    if k == "hermite":  # 28 steps per particle in 1/8 of a time unit at 16384 particles
        return dict(bytes=176.0 * case["n"],
                    flops=60.0 * case["n"] ** 2 * (1 + 225 * case["t"] * (case["n"] / 16384) ** (1 / 3)))
    if k == "clusters":  # moments of a log-uniform size
        lo, hi = case["nmin"], case["nmax"]
        ln = math.log(hi / lo)
        n1, n2 = (hi - lo) / ln, (hi ** 2 - lo ** 2) / (2 * ln)
        return dict(bytes=112.0 * case["ncl"] * n1, flops=60.0 * case["ncl"] * n2)
    n = case.get("n")
    if k == "treepm_lists":  # positions in and out, indices, about 44 list entries a particle
        return dict(bytes=(24.0 + 24.0 + 8.0 + 4.0 * 44) * n, flops=0.0)
    if k in ("treepm_table", "treepm_mlp"):
        # the network: 16 + 256 + 16 multiply-adds and 32 activations of 3 flops
        each = 38.0 if k == "treepm_table" else 38.0 + 2 * 288 + 3 * 32
        return dict(bytes=(16.0 + 24.0 + 4.0 * 44 + (24.0 if case["origin"] else 0.0)) * n,
                    flops=each * treepm_pairs(n))
    if k == "pm":  # particles in, accelerations out; four FFTs
        m3 = case["mesh"] ** 3
        return dict(bytes=56.0 * n, flops=4 * 2.5 * m3 * math.log2(m3) + 27 * 10.0 * n)
    # 8.6 particle and 19.2 cell list entries a particle at 2^21 particles and
    # theta = 0.5, groups of about 180 particles
    grow = math.log2(n) / 21 * (0.5 / case["theta"]) ** 2
    if k == "bh_lists":
        return dict(bytes=(32.0 + 36.0 + 4.0 * 27.8 * grow) * n, flops=0.0)
    return dict(bytes=(48.0 + 4.0 * 27.8 * grow) * n,
                flops=(38.0 * 1574 + 71.0 * 3004) * grow * n)


# ------------------------------------------------------------------ 64 bits
def s2(r, a):
    """Force per unit separation between two S2 spheres of diameter a
    (Hockney & Eastwood), numpy or torch."""
    e = 2.0 * r / a
    w = np.where if isinstance(e, np.ndarray) else torch.where
    lo = (224 + e * e * (-224 + e * (70 + e * (48 - 21 * e)))) * 2 / (35 * a ** 3)
    f = w(e > 0.5, e, e * 0 + 1)
    mid = (12 / (f * f) - 224 + f * (896 + f * (-840 + f * (224 + f * (70 + f * (7 * f - 48)))))
           ) * 2 / (35 * f * a ** 3)
    g = w(e > 1.5, r, r * 0 + a)
    return w(e < 1, lo, w(e < 2, mid, 1 / g ** 3))


def table_shape(n, frc, order):
    """The tabulated shape as a function of r^2: value and slope (or a
    quadratic) between the float ticks of s = 2 + r^2 (s_max - 2) / r_cut^2."""
    pp, pm = split_of(n)
    scale = (65536 * (2 - 0.5 ** frc) - 2) / pm ** 2
    q = 1 << frc
    s = np.array([2.0 ** (1 + k // q) * (1 + (k % q) / q) for k in range(16 * q + 1)])
    f = lambda v: s2(np.sqrt((v - 2) / scale), pp) - s2(np.sqrt((v - 2) / scale), pm)  # noqa: E731
    h, f0, f1 = np.diff(s), f(s[:-1]), f(s[1:])
    fm = f(s[:-1] + h / 2)
    c2 = 2 * (f1 - 2 * fm + f0) / h ** 2 if order == 2 else 0 * h
    c1 = (f1 - f0) / h - c2 * h
    c1[-1] = c2[-1] = 0
    s, c0, c1, c2 = (dev(v) for v in (s[:-1], f0, c1, c2))

    def shape(r2):
        v = 2 + r2 * scale
        mant, e = torch.frexp(v)
        k = ((e - 2) * q + torch.floor((2 * mant - 1) * q).to(e.dtype)).clamp(max=16 * q - 1).long()
        d = torch.minimum(v, s[-1]) - s[k]
        return c0[k] + d * (c1[k] + d * c2[k])

    return shape


def network_shape(n):
    """f(r^2) of the network: 1 / r^3 (the S2 core inside eps_PP) less the
    network's unit shape at eps_PM, 0 beyond it."""
    pp, pm = split_of(n)
    p = dev(network())

    def unit(u):
        h = torch.tanh((2 * u[..., None] - 1) * p[:16] + p[16:32])
        h = torch.tanh(h.reshape(-1, 16) @ p[32:288].reshape(16, 16).T.contiguous() + p[288:304])
        return (h @ p[304:320] + p[320]).reshape(u.shape)

    def shape(r2):
        flat = r2.reshape(-1)
        out = torch.zeros_like(flat)
        at = ((flat > 0) & (flat < pm * pm)).nonzero()[:, 0]
        r = flat[at].sqrt()
        near = torch.where(r < pp, unit((r / pp).clamp(max=1)) / pp ** 3, 1 / r ** 3)
        out[at] = near - unit(r / pm) / pm ** 3
        return out.reshape(r2.shape)

    return shape


def direct(xi, xj, m, e2, step=1024):
    """acc and + sum m / r of xi against xj; e2 a number or [ni, nj]-broadcast."""
    acc, pot = torch.empty_like(xi), torch.empty_like(xi[:, 0])
    for a in range(0, len(xi), step):
        d = xj[None] - xi[a:a + step, None]
        r = ((d * d).sum(-1) + e2).rsqrt()
        pot[a:a + step] = (m * r).sum(1)
        acc[a:a + step] = ((m * r ** 3)[..., None] * d).sum(1)
    return acc, pot


def hermite_direct(xi, vi, xj, vj, m, e2, self_of, step=1024):
    """acc, jerk and - sum m / r, the pair (i, self_of[i]) left out."""
    acc, jrk, pot = torch.empty_like(xi), torch.empty_like(xi), torch.empty_like(xi[:, 0])
    for a in range(0, len(xi), step):
        s = slice(a, a + step)
        d, dv = xj[None] - xi[s, None], vj[None] - vi[s, None]
        r = ((d * d).sum(-1) + e2).rsqrt()
        r[torch.arange(len(r), device="cuda"), self_of[s]] = 0
        mr3 = m * r ** 3
        beta = -3 * (d * dv).sum(-1) * r * r
        acc[s] = (mr3[..., None] * d).sum(1)
        jrk[s] = (mr3[..., None] * (dv + beta[..., None] * d)).sum(1)
        pot[s] = -(m * r).sum(1)
    return acc, jrk, pot


def groups(h, g):
    i = h["ilist"][h["ioff"][g]:h["ioff"][g] + h["icnt"][g]]
    j = h["jlist"][h["joff"][g]:h["joff"][g] + h["jcnt"][g]]
    return i, j


def mesh_force(x, m, M, a):
    """TSC assignment, FFT, Green's function of the S2 shape of diameter a
    with the window squared divided out, spectral gradient (Nyquist modes
    dropped), TSC interpolation."""
    u = x * M
    g = torch.floor(u + 0.5)
    d = u - g
    w = torch.stack([0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2], -1)
    g = g.long()
    terms = []
    for i in range(27):
        o = (i // 9, i // 3 % 3, i % 3)
        at = [(g[:, q] + o[q] - 1) % M for q in range(3)]
        terms.append(((at[0] * M + at[1]) * M + at[2], w[:, 0, o[0]] * w[:, 1, o[1]] * w[:, 2, o[2]]))
    rho = torch.zeros(M ** 3, dtype=torch.float64, device="cuda")
    for at, q in terms:
        rho.index_add_(0, at, m * q * M ** 3)
    n = torch.fft.fftfreq(M, 1 / M, dtype=torch.float64, device="cuda")
    nz = torch.arange(M // 2 + 1, dtype=torch.float64, device="cuda")
    k = [2 * math.pi * v for v in torch.meshgrid(n, n, nz, indexing="ij")]
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    win = torch.ones_like(k2)
    for v in k:
        win *= torch.sinc(v / (2 * math.pi * M)) ** 3
    q = k2.sqrt() * a / 2
    safe = q.clamp(min=1e-3)
    form = torch.where(q > 1e-3, 12 / safe ** 4 * (2 - 2 * torch.cos(safe) - safe * torch.sin(safe)),
                       1 - q * q / 15)
    green = -4 * math.pi * form ** 2 / (k2.clamp(min=1) * win ** 2)
    green[0, 0, 0] = 0
    green[M // 2], green[:, M // 2], green[:, :, M // 2] = 0, 0, 0
    phi = torch.fft.rfftn(rho.reshape(M, M, M)) * green
    acc = torch.zeros_like(x)
    for axis in range(3):
        f = torch.fft.irfftn(-1j * k[axis] * phi, s=(M, M, M)).reshape(-1)
        for at, q in terms:
            acc[:, axis] += q * f[at]
    return acc


def exact(case, seed):
    k = case["kind"]
    if k == "g5_host":
        m, x, _ = ics.plummer(case["n"], seed)
        a, p = direct(dev(x), dev(x), dev(m), case["eps"] ** 2)
        return a.cpu().numpy(), p.cpu().numpy()
    if k == "g5_dev":
        xi, xj, e2j = (None if v is None else dev(v).double() for v in halves(case, seed))
        e2 = case["eps"] ** 2
        return direct(xi[:, :3], xj[:, :3], xj[:, 3], e2 if e2j is None else e2 + e2j)
    if k in ("g6_host", "g6_dev"):
        t, x, v, sel = block(case, seed)
        xj, vj = predicted(case["nj"], t)
        out = hermite_direct(dev(x), dev(v), dev(xj), dev(vj), dev(model(case["nj"])[0]),
                             case["eps"] ** 2, dev(sel).long(), 512)
        if k == "g6_host":
            out = tuple(v.cpu().numpy() for v in out)
        nn = dict(nnb=None, rnnb=None) if case.get("nn", True) else {}
        return dict(acc=out[0], jrk=out[1], pot=out[2], **nn)
    if k == "clusters":
        size, coff, x, v, m, e2 = star_clusters(case, seed)
        x, v, m = dev(x), dev(v), dev(m)
        out = [torch.empty_like(x), torch.empty_like(x), torch.empty_like(m)]
        for c in range(len(size)):
            q = slice(int(coff[c]), int(coff[c + 1]))
            got = hermite_direct(x[q], v[q], x[q], v[q], m[q], float(e2[c]),
                                 torch.arange(int(size[c]), device="cuda"), 4096)
            for o, r in zip(out, got):
                o[q] = r
        return tuple(out)
    if k in ("treepm_table", "treepm_mlp"):
        m, _, DL = treepm_lists_of(case["n"], seed)
        h = DL.host()
        shape = (network_shape(case["n"]) if k == "treepm_mlp"
                 else table_shape(case["n"], case["frc"], case["order"]))
        x, mj = dev(h["pos"]), dev(m[h["src"]])
        ilist, jlist = dev(h["ilist"]).long(), dev(h["jlist"]).long()
        acc = torch.zeros((case["n"], 3), dtype=torch.float64, device="cuda")
        for g in range(len(h["ioff"])):
            i, j = groups(dict(h, ilist=ilist, jlist=jlist), g)
            d = x[j][None] - x[i][:, None]
            acc[i] = ((mj[j] * shape((d * d).sum(-1)))[..., None] * d).sum(1)
        return acc
    if k == "pm":
        m, x = ics.clumpy_box(case["n"], seed)
        return mesh_force(dev(x), dev(m), case["mesh"], 3.0 / case["mesh"])
    if k == "bh_force":
        m, _, DL = bh_lists_of(case, seed)
        h = DL.host()
        x, mj, cells = dev(h["pos"]), dev(m[h["src"]]), dev(h["cells"])
        lists = {q: dev(h[q]).long() for q in ("ilist", "jlist", "clist")}
        acc = torch.zeros((case["n"], 3), dtype=torch.float64, device="cuda")
        pot = torch.zeros(case["n"], dtype=torch.float64, device="cuda")
        e2 = case["eps"] ** 2
        for g in range(len(h["ioff"])):
            i, j = groups(dict(h, **lists), g)
            a, p = direct(x[i], x[j], mj[j], e2)
            c = cells[lists["clist"][h["coff"][g]:h["coff"][g] + h["ccnt"][g]]]
            d = c[None, :, :3] - x[i][:, None]
            r = ((d * d).sum(-1) + e2).rsqrt()
            dx, dy, dz = d.unbind(-1)
            xx, xy, xz, yy, yz, zz = c[:, 4:].T
            qd = torch.stack([xx * dx + xy * dy + xz * dz, xy * dx + yy * dy + yz * dz,
                              xz * dx + yz * dy + zz * dz], -1)
            mono, quad = c[:, 3] * r, 0.5 * (qd * d).sum(-1) * r ** 5
            acc[i] = a + (((mono + 5 * quad) * r * r)[..., None] * d - r[..., None] ** 5 * qd).sum(1)
            pot[i] = p + (mono + quad).sum(1)
        return acc, pot
    # an integration diverges from any other arithmetic's; lists are decisions
    return None
