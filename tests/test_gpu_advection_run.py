"""AdvectionSolver.run against the step entry points it replaces (bit for bit)."""
import numpy as np
import pytest

from conftest import gpu_available, make_tet_domain, make_tri_domain
from test_gpu_mixed_meshes import tri_quad_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _domain(kind):
    if kind == "mixed":
        return tri_quad_domain(13, 9, 1., 1.)
    if isinstance(kind, int):
        return make_tet_domain(kind)
    return make_tri_domain(*kind)


def _bits(a, b):
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("kind,order,nsteps", [((3, 2), 1, 1), ((3, 2), 2, 2), ((17, 9), 1, 5), ((17, 9), 2, 4),
                                               ((17, 9), 1, 6), ((41, 37), 1, 9), ((41, 37), 1, 12),
                                               ("mixed", 1, 7), (3, 1, 8),
                                               ("mixed", 1, 3), ("mixed", 2, 3), (2, 1, 3), (2, 2, 2), (4, 2, 3)])
def test_advection_run_equals_the_steps(kind, order, nsteps):
    import torch
    from manapy_amd import AdvectionSolver, Struct, Variable, _lib
    from manapy_amd.device import stream_ptr
    d = _domain(kind)
    C, F, dim = int(d.nbcells), int(d.nbfaces), int(d.dim)
    rng = np.random.default_rng(C + 7 * order)
    var = Variable(domain=d)
    vel = [Variable(domain=d) for _ in range(dim)]
    w0 = torch.as_tensor(rng.normal(size=C), device="cuda")
    var.cell.copy_(w0)
    for v in vel:
        u = rng.normal(size=F)
        u[rng.random(F) < .2] = 0.  # faces without flow, both signs of zero
        u[rng.random(F) < .1] = -0.
        v.face[:] = torch.as_tensor(u, device="cuda")
        v.interpolate_facetocell()
    sol = AdvectionSolver(var, vel=tuple(vel), conf=Struct(order=order, cfl=.4))
    t = sol.run(nsteps)

    m, s = d.device_mesh, stream_ptr()
    u = [x.cell for x in (sol.u, sol.v, sol.w)] + [x.face for x in (sol.u, sol.v, sol.w)]
    dt0, ring = torch.zeros(1, dtype=torch.float64, device="cuda"), torch.zeros(4, dtype=torch.float64, device="cuda")
    _lib.call("mfv_time_step", m.ptr, *[x.data_ptr() for x in u[:3]], .4, dt0.data_ptr(), None, s)
    _lib.call("mfv_dt_ring_init", ring.data_ptr(), dt0.data_ptr(), s)
    a, b = w0.clone(), torch.empty_like(w0)
    scratch = torch.zeros((dim + 1) * C, dtype=torch.float64, device="cuda")
    for k in range(nsteps):
        _lib.call("mfv_advection_step", m.ptr, a.data_ptr(), b.data_ptr(), *[x.data_ptr() for x in u], .4, order,
                  ring.data_ptr(), k, scratch.data_ptr(), s)
        a, b = b, a
    _bits(var.cell, a)
    _bits(sol._clock.ring, ring)
    assert t == float(ring[3])
