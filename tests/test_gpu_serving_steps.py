"""The time steps that the solver's products take by themselves (mfv_krylov_fused_tick with
steps_left) against the same steps driven from the host: mfv_advection_step into b, the first guess
x = b, one solve, step by step (bit for bit)."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available, make_tri_domain
from test_gpu_mixed_meshes import tri_quad_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _host_driven(d, u0, velocity, D, nsteps, width):
    import torch
    from manapy_amd import _lib
    from manapy_amd.device import stream_ptr
    from manapy_amd.krylov import EllBatch
    C, F = int(d.nbcells), int(d.nbfaces)
    m, s, P = d.device_mesh, stream_ptr(), lambda t: t.data_ptr()
    z = lambda n: torch.zeros(n, dtype=torch.float64, device="cuda")
    uf, vf, wf, uc, vc, wc = z(F) + velocity[0], z(F) + velocity[1], z(F), z(C), z(C), z(C)
    _lib.call("mfv_facetocell", m.ptr, P(uf), P(uc), s)
    _lib.call("mfv_facetocell", m.ptr, P(vf), P(vc), s)
    dt, ring, h = z(1), z(4), ctypes.c_double(0.)
    _lib.call("mfv_time_step", m.ptr, P(uc), P(vc), P(wc), .8, P(dt), ctypes.byref(h), s)
    _lib.call("mfv_dt_ring_init", P(ring), P(dt), s)
    a = EllBatch((C + 63) // 64, max_inst=1, width=width)
    i = a.alloc(C)
    a.assemble_diamond(i, d.device_diamond, torch.zeros(int(d.nbnodes), dtype=torch.uint8, device="cuda"),
                       torch.full((F,), -1, dtype=torch.int32, device="cuda"))
    a.publish()
    a.configure(i, 1., -h.value * D, tol=1e-10, tol_in=1e-3)
    a.x[:C] = torch.as_tensor(u0, device="cuda")
    for k in range(nsteps):
        _lib.call("mfv_advection_step", m.ptr, P(a.x), P(a.b), P(uc), P(vc), P(wc), P(uf), P(vf), P(wf), .8, 1,
                  P(ring), k, None, s)
        a.x[:C] = a.b[:C]
        a.status[i] = _lib.KS_START
        assert a.run([i], n_iter=5)[0] == _lib.KS_DONE
    return a.x[:C].cpu().numpy(), int(a.scalars(i)[_lib.KS_ITTOT])


MESHES = [lambda: make_tri_domain(2, 2), lambda: make_tri_domain(17, 9), lambda: tri_quad_domain(13, 9, 1., 1.),
          lambda: make_tri_domain(70, 61)]


@pytest.mark.parametrize("n_iter,graph", [(1, False), (6, True)])
@pytest.mark.parametrize("slots", [1, 4])  # one request after the other in the same slot, or all together
def test_steps_on_the_device(n_iter, graph, slots):
    from manapy_amd.serving import AdvDiffRequest, ServingEngine, PHASE_DONE
    reqs, want = [], []
    for k, make in enumerate(MESHES):
        d = make()
        rng = np.random.default_rng(k)
        u0, vel, D, n = rng.random(int(d.nbcells)), (1., -.4 + .3 * k), 10. ** -(1 + k % 3), 1 + k
        want.append(_host_driven(d, u0, vel, D, n, 16))
        d._device_mesh = d._device_diamond = None
        reqs.append(AdvDiffRequest(k, d, u0, velocity=vel, D=D, nsteps=n))
    done = ServingEngine(max_cells=1 << 14, max_inst=slots, n_iter=n_iter, graph=graph).run(reqs)
    assert sorted(r.rid for r in done) == list(range(len(MESHES)))
    for r in done:
        assert r.phase == PHASE_DONE and r.step == r.nsteps
        np.testing.assert_array_equal(r.result, want[r.rid][0])
        assert r.iterations == want[r.rid][1]


def test_failing_step_is_reported():
    from manapy_amd.serving import AdvDiffRequest, ServingEngine, PHASE_FAILED
    d = make_tri_domain(9, 7)
    u0 = np.ones(int(d.nbcells))
    u0[3] = np.nan
    r = ServingEngine(max_cells=1 << 12, max_inst=2).run([AdvDiffRequest(0, d, u0, nsteps=3)])[0]
    assert r.phase == PHASE_FAILED and "step 0" in r.error
