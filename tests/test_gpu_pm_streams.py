"""Mesh-force calls queued on several streams without a synchronisation between
them: they share one workspace, so each must wait for the one before it."""
import numpy as np
import pytest

import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(200000, 64), (3000, 64)],             # sorted, direct; the same mesh
    [(200000, 64), (150000, 64), (60000, 64)],  # brick tables of different particles
    [(100000, 48), (100000, 64), (500, 96)],    # other meshes: new plans and buffers
])
def test_calls_on_several_streams_do_not_overlap(sizes):
    import pgamd
    import torch
    T = pgamd.G5Table()
    work = []
    for k, (n, mesh) in enumerate(sizes):
        m, x = ics.clumpy_box(n, 50 + k)
        work.append([n, mesh, torch.from_numpy(x).cuda(), torch.from_numpy(m).cuda(),
                     torch.empty((n, 3), dtype=torch.float64, device="cuda")])

    def call(w, stream):
        n, mesh, x, m, acc = w
        assert T.lib.pg5t_pm_force(n, x.data_ptr(), m.data_ptr(), mesh, 3.0 / mesh,
                                   acc.data_ptr(), stream) == 0

    want = []
    for w in work:
        torch.cuda.synchronize()
        call(w, None)
        torch.cuda.synchronize()
        want.append(w[4].cpu().numpy())
    streams = [torch.cuda.Stream() for _ in work]
    handles = [s.cuda_stream for s in streams[:-1]] + [None]  # the last on the library's own
    for shift in range(2 * len(work)):
        for w in work:
            w[4].fill_(7.0)
        torch.cuda.synchronize()
        for _ in range(3):
            for k, w in enumerate(work):
                call(w, handles[(k + shift) % len(work)])
        torch.cuda.synchronize()
        for w, a in zip(work, want):
            np.testing.assert_array_equal(w[4].cpu().numpy(), a)



@pytest.mark.parametrize("first", ["caller", "library"])
@pytest.mark.parametrize("n", [0, 1, 30000])
def test_a_call_runs_after_the_one_before_it(n, first):
    """A long call, then a short one on another stream: what that stream does next
    finds the long call's result complete."""
    import ctypes

    import pgamd
    import torch
    T = pgamd.G5Table()
    mesh, long = 128, 1 << 20
    m, x = ics.clumpy_box(long, 3)
    x, m = torch.from_numpy(x).cuda(), torch.from_numpy(m).cuda()
    acc, other, own = (torch.empty((k, 3), dtype=torch.float64, device="cuda")
                       for k in (long, long, max(n, 1)))
    T.lib.pg5t_dev_stream.restype, T.lib.pg5t_dev_stream.argtypes = ctypes.c_void_p, [ctypes.c_int]
    a = torch.cuda.Stream().cuda_stream if first == "caller" else T.lib.pg5t_dev_stream(0)
    b = torch.cuda.Stream()

    def call(k, out, stream):
        assert T.lib.pg5t_pm_force(k, x.data_ptr(), m.data_ptr(), mesh, 3.0 / mesh, out.data_ptr(),
                                   stream) == 0

    call(long, acc, a)
    torch.cuda.synchronize()
    want = acc.clone()
    for _ in range(10):
        acc.fill_(7.0)
        torch.cuda.synchronize()
        for out in (other, other, acc):
            call(long, out, a)
        call(n, own, b.cuda_stream)
        with torch.cuda.stream(b):
            got = acc.clone()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
