"""ShallowWaterSolver.run (flux='srnh') with its fused steps against the sequence of stepper,
compute_fluxes and compute_new_val (bit for bit), with every array that the sequence leaves: step
counts that run none, some and an even or odd rest of them, a part of a wave, more than the 1024
partials that a step folds itself, and boundary values of every kind."""
import numpy as np
import pytest

from conftest import gpu_available, make_tri_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

MIXED = {"in": "dirichlet", "out": "neumannNH", "upper": "nonslip", "bottom": "neumann"}


def _solver(d, order, quirk, mixed):
    import torch
    from manapy_amd import ShallowWaterSolver, Struct, Variable
    C = int(d.nbcells)
    rng = np.random.default_rng(C + order)
    wall = dict.fromkeys(("in", "out", "upper", "bottom"), "nonslip")
    kw = lambda v: dict(BC=MIXED, values={"in": v, "out": .1}) if mixed else {}  # noqa: E731
    h, hc, Z = Variable(domain=d, **kw(1.4)), Variable(domain=d, **kw(.14)), Variable(domain=d)
    hu, hv = Variable(domain=d, BC=wall), Variable(domain=d, BC=wall)
    for v, a in ((h, 1. + rng.random(C)), (hu, .1 * rng.normal(size=C)), (hv, .1 * rng.normal(size=C)),
                 (hc, .1 * rng.random(C)), (Z, .1 * rng.random(C))):
        v.cell[:] = torch.as_tensor(a, device="cuda")
    return ShallowWaterSolver(h=h, hvel=(hu, hv), hc=hc, Z=Z,
                              conf=Struct(order=order, cfl=.8, flux="srnh", quirk=quirk))


@pytest.mark.parametrize("size,order,nsteps,quirk,mixed",
                         [((3, 2), 2, 1, True, False), ((3, 2), 1, 3, True, True), ((17, 9), 2, 2, False, True),
                          ((17, 9), 2, 4, True, True), ((17, 9), 1, 7, False, False), ((190, 180), 2, 3, True, False)])
def test_run_equals_the_sequence(size, order, nsteps, quirk, mixed):
    d = make_tri_domain(*size, 10., 10. * size[1] / size[0])
    a, b = _solver(d, order, quirk, mixed), _solver(d, order, quirk, mixed)
    t, want = a.run(nsteps), 0.
    for _ in range(nsteps):
        want += b.stepper()
        b.compute_fluxes()
        b.compute_new_val()
    assert t == want and a.dt == b.dt
    for name in a.varbs:
        x, y = a.varbs[name], b.varbs[name]
        for k in ("cell", "ghost", "convective", "source", "gradcellx", "gradcelly", "psi"):
            np.testing.assert_array_equal(getattr(x, k).cpu().numpy(), getattr(y, k).cpu().numpy(), "%s.%s" % (name, k))
