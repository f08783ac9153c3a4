"""The dt that a stepper returns: the device's own value, from any thread and stream, also behind a
long queue; refused under capture."""
import ctypes
import threading

import numpy as np
import pytest

from conftest import gpu_available, make_tet_domain, make_tri_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _setup(d, seed):
    import torch
    rng = np.random.default_rng(seed)
    C = int(d.nbcells)
    u = [torch.as_tensor(rng.normal(size=C), device="cuda") for _ in range(3)]
    return u, torch.zeros(1, dtype=torch.float64, device="cuda")


def _dt(m, u, dt_dev, stream):
    from manapy_amd import _lib
    h = ctypes.c_double(-1.)
    _lib.call("mfv_time_step", m.ptr, *[x.data_ptr() for x in u], .4, dt_dev.data_ptr(), ctypes.byref(h), stream)
    return h.value


def _expected(d, u):
    n, fid = d.faces.normal, d.cells.faceid
    lam = np.zeros(int(d.nbcells))
    v = np.stack([x.cpu().numpy() for x in u], axis=1)
    for j in range(fid.shape[1] - 1):
        ok = j < fid[:, -1]
        f = np.where(ok, fid[:, j], 0)
        lam += np.where(ok, np.abs((v * n[f][:, :3]).sum(1)), 0.)
    return min(1e6, float((.4 * d.cells.volume / lam).min()))


# one wave, a block's remainder, more partials than threads of the fold (1024 waves = 65 536 cells)
@pytest.mark.parametrize("make,size", [(make_tri_domain, (2, 1)), (make_tri_domain, (13, 11)),
                                       (make_tri_domain, (200, 170)), (make_tet_domain, (3,))])
def test_value_on_host_and_device(make, size):
    from manapy_amd.device import stream_ptr
    d = make(*size)
    u, dev = _setup(d, 3)
    h = _dt(d.device_mesh, u, dev, stream_ptr())
    assert h == float(dev)
    np.testing.assert_allclose(h, _expected(d, u), rtol=1e-13)
    u[0].zero_(), u[1].zero_(), u[2].zero_()  # no velocity: the reference's start value
    assert _dt(d.device_mesh, u, dev, stream_ptr()) == 1e6 == float(dev)


def test_behind_a_long_queue():
    import torch
    from manapy_amd.device import stream_ptr
    d = make_tri_domain(13, 11)
    u, dev = _setup(d, 4)
    want = _dt(d.device_mesh, u, dev, stream_ptr())
    a = torch.zeros(1 << 28, device="cuda")
    for _ in range(120):  # about 0.3 ms each, more than the call looks at the value by itself
        a.add_(1.)
    assert _dt(d.device_mesh, u, dev, stream_ptr()) == want


def test_threads_on_their_own_streams():
    import torch
    d = make_tri_domain(41, 37)
    m = d.device_mesh
    sets = [_setup(d, 10 + k) for k in range(4)]
    want = [_expected(d, u) for u, _ in sets]
    torch.cuda.synchronize()
    got = [[] for _ in sets]

    def work(k):
        s = torch.cuda.Stream()
        for _ in range(50):
            got[k].append(_dt(m, sets[k][0], sets[k][1], s.cuda_stream))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for k in range(4):
        assert len(set(got[k])) == 1
        np.testing.assert_allclose(got[k][0], want[k], rtol=1e-13)


def test_refused_under_capture():
    import torch
    from manapy_amd import _lib
    from manapy_amd.device import stream_ptr
    d = make_tri_domain(13, 11)
    u, dev = _setup(d, 5)
    s = torch.cuda.Stream()
    _dt(d.device_mesh, u, dev, s.cuda_stream)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        g.capture_begin()
        try:
            with pytest.raises(_lib.MfvError, match="captured"):
                _dt(d.device_mesh, u, dev, stream_ptr())
        finally:
            g.capture_end()
    torch.cuda.synchronize()
    assert _dt(d.device_mesh, u, dev, stream_ptr()) == float(dev)


def _time_steps(d, u, dev, form, stream):
    """(name, call) of the four time steps with a host dt, in one of their two forms."""
    import torch
    from manapy_amd import _lib
    m, P = d.device_mesh, lambda *ts: [t.data_ptr() for t in ts]
    h = ctypes.c_double(-1.)

    def call(name, *args):
        _lib.call(name + form, m.ptr, *args, dev.data_ptr(), ctypes.byref(h), stream)
        return h.value

    out = [("mfv_time_step", lambda: call("mfv_time_step", *P(*u), .4)),
           ("mfv_time_step_diffusion", lambda: call("mfv_time_step_diffusion", *P(*u), .4, .1, .1, .1))]
    if m.dim == 2:
        pos = u[0].abs() + 1.
        out.append(("mfv_time_step_sw", lambda: call("mfv_time_step_sw", *P(pos, u[1], u[2]), .4, 9.81, 0., 0.)))
    else:
        U = torch.stack([u[0].abs() + 1., u[0].abs() + 2., u[0], u[1], u[2], u[0].abs() + 9.])
        out.append(("mfv_euler3d_time_step", lambda: call("mfv_euler3d_time_step", U.data_ptr(), .4, 1.4)))
    return out


@pytest.mark.parametrize("make,size", [(make_tri_domain, (200, 170)), (make_tet_domain, (6,))])
def test_the_stream_is_idle_after_a_host_dt(make, size):
    """include/mfv.h: a call with a *_host output synchronises its stream."""
    import torch
    d = make(*size)
    u, dev = _setup(d, 6)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    for name, call in _time_steps(d, u, dev, "", s.cuda_stream):
        for _ in range(50):
            call()
            assert s.query(), name


@pytest.mark.parametrize("make,size", [(make_tri_domain, (200, 170)), (make_tet_domain, (6,))])
def test_the_polled_dt_is_seen_on_any_stream(make, size):
    """The polled form: dt_dev and what the stream held before it are there for work that the caller
    starts next on another stream, with no synchronisation between."""
    import torch
    d = make(*size)
    u, dev = _setup(d, 7)
    torch.cuda.synchronize()
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    for name, call in _time_steps(d, u, dev, "_polled", s.cuda_stream):
        idle = dict(_time_steps(d, u, dev, "", s.cuda_stream))[name]()
        before = torch.zeros(1 << 20, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        for k in range(1, 51):
            with torch.cuda.stream(s):
                before.fill_(k)
                dev.fill_(-1.)
            got = call()
            with torch.cuda.stream(other):
                seen, sees = dev.clone(), before.clone()
            other.synchronize()
            assert got == idle == float(seen) and bool((sees == k).all()), (name, k)
        s.synchronize()
