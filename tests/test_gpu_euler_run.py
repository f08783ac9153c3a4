"""EulerSolver3D.run on Morton-ordered face tiles against the per-cell fused steps in the mesh's own
order (bit for bit): 48 cells (part of a wave), several tiles with remainders, 63 888 cells (999 partials, the
most that the next step folds is 1024) and 73 002 (a fold launch a step)."""
import numpy as np
import pytest

from conftest import gpu_available, make_tet_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("n,nsteps,quirk", [(2, 2, False), (2, 1, True), (5, 4, True), (5, 3, False), (22, 3, False),
                                            (23, 2, False)])
def test_run_equals_the_fused_steps(n, nsteps, quirk):
    import torch
    from manapy_amd import EulerSolver3D
    d = make_tet_domain(n)
    C = int(d.nbcells)
    rng = np.random.default_rng(n)
    U = np.zeros((6, C))
    U[0], U[1] = 1. + rng.random(C), 1. + rng.random(C)
    U[2:5] = .2 * rng.normal(size=(3, C))
    U[5] = .5 * (U[2:5] ** 2).sum(0) / U[0] + U[1] / .4
    got, want = (EulerSolver3D(d, U, cfl=.8, quirk=quirk) for _ in range(2))
    t = got.run(nsteps)
    assert d.device_mesh._euler_run.tiles is not None
    assert t == want.run(nsteps, packed=False) and got.dt == want.dt
    np.testing.assert_array_equal(got.U.cpu().numpy(), want.U.cpu().numpy())
    np.testing.assert_array_equal(got._clock.ring.cpu().numpy(), want._clock.ring.cpu().numpy())
    got.run(0)  # no step: the records' way there and back leaves the state
    np.testing.assert_array_equal(got.U.cpu().numpy(), want.U.cpu().numpy())
