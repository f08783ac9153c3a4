"""ShallowWaterSolver.run (flux='rusanov') against the step entry points it replaces (bit for bit)."""
import numpy as np
import pytest

from conftest import gpu_available, make_tri_domain
from test_gpu_mixed_meshes import tri_quad_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

WALLS = {"in": "nonslip", "out": "nonslip", "upper": "nonslip", "bottom": "nonslip"}


def _domain(kind):
    if kind == "mixed":
        return tri_quad_domain(13, 9, 1., 1.)
    return make_tri_domain(*kind)


def _bits(a, b):
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


# 12 cells (part of a wave), one block's worth, 16.4k cells (above the small-mesh rule), 65 536 cells
# (1024 partials, the last folded by the next step) and 66 048 (a fold launch each)
@pytest.mark.parametrize("kind,order,nsteps", [((3, 2), 2, 1), ((3, 2), 1, 4), ((11, 7), 2, 5), ((91, 91), 2, 2),
                                               ((256, 128), 2, 3), ((258, 128), 2, 3), ("mixed", 1, 3),
                                               ("mixed", 2, 4)])
def test_sw_run_equals_the_two_kernel_steps(kind, order, nsteps):
    import torch
    from manapy_amd import ShallowWaterSolver, Struct, Variable, _lib
    from manapy_amd.device import DeviceMesh, SwPacked, stream_ptr
    from manapy_amd.renumber import renumbered
    d = _domain(kind)
    C = int(d.nbcells)
    rng = np.random.default_rng(C + order)
    h, hu, hv = Variable(domain=d), Variable(domain=d, BC=WALLS), Variable(domain=d, BC=WALLS)
    Z = Variable(domain=d)
    dev = lambda a: torch.as_tensor(a, device="cuda")
    for var, a in ((h, 1. + rng.random(C)), (hu, .1 * rng.normal(size=C)), (hv, .1 * rng.normal(size=C)),
                   (Z, .1 * rng.random(C))):
        var.cell[:] = dev(a)
    start = [v.cell.clone() for v in (h, hu, hv)]
    sol = ShallowWaterSolver(h=h, hvel=(hu, hv), Z=Z, conf=Struct(order=order, cfl=.8, flux="rusanov"))
    t = sol.run(nsteps)

    r = renumbered(d)
    rm, perm = DeviceMesh(r), torch.as_tensor(r.perm, device="cuda")
    p = SwPacked(rm)
    p.pack(rm, *[x[perm] for x in start], Z.cell[perm], sol._zgrad[:, perm].contiguous(), order)
    ring, dt0 = torch.zeros(4, dtype=torch.float64, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    m = d.device_mesh
    _lib.call("mfv_time_step_sw", m.ptr, *[x.data_ptr() for x in start], .8, 9.81, 0., 0., dt0.data_ptr(), None,
              stream_ptr())
    _lib.call("mfv_dt_ring_init", ring.data_ptr(), dt0.data_ptr(), stream_ptr())
    for k in range(nsteps):
        _lib.call("mfv_sw_recon", rm.ptr, p.ptr, order, stream_ptr())
        _lib.call("mfv_sw_flux_packed", rm.ptr, p.ptr, 9.81, .8, ring.data_ptr(), k, stream_ptr())
    for v, col in ((h, 5), (hu, 3), (hv, 4)):
        _bits(v.cell[perm], p.cellrec[:, col])
    _bits(sol._clock.ring, ring)
    assert t == float(ring[3])


def test_sw_solvers_of_one_mesh_share_tables_not_states():
    import torch
    from manapy_amd import ShallowWaterSolver, Struct, Variable
    d = make_tri_domain(9, 8)
    C = int(d.nbcells)

    def solver(seed):
        rng = np.random.default_rng(seed)
        h, hu, hv = Variable(domain=d), Variable(domain=d, BC=WALLS), Variable(domain=d, BC=WALLS)
        Z = Variable(domain=d)
        h.cell[:] = torch.as_tensor(1. + rng.random(C), device="cuda")
        Z.cell[:] = torch.as_tensor(.1 * rng.random(C), device="cuda")
        return ShallowWaterSolver(h=h, hvel=(hu, hv), Z=Z, conf=Struct(order=2, cfl=.8, flux="rusanov"))

    alone = solver(1)
    alone.run(3)
    alone.run(3)
    a, b = solver(1), solver(2)
    a.run(3)
    b.run(3)
    a.run(3)
    _bits(a.h.cell, alone.h.cell)
    assert a._packed.tables is b._packed.tables and a._packed.cfrec is not b._packed.cfrec
