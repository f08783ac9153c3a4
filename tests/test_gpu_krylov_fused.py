"""The two-launch BiCGStab tick: chunk lists (CPU) and solves at the sizes where its partition
changes (one row, a slice, a block's four slices, two slices per wave), against the FP64
residual formed from the matrix itself and against the eight-launch tick."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available, make_tri_domain


def _span(ns):
    return 4 * ((ns + 2047) // 2048)


def test_chunk_list_covers_every_slice_once():
    from manapy_amd.krylov import chunk_list
    ranges = [(3, 0, 1), (0, 1, 4), (7, 5, 5), (1, 10, 2048), (2, 2058, 2049), (5, 4107, 70000)]
    ch = chunk_list(ranges)
    assert ch.dtype == np.int32 and ch.shape[1] == 4
    for inst, s0, ns in ranges:
        c = ch[ch[:, 0] == inst]
        n = c[:, 2] >> 16
        assert np.all(c[:, 1] == s0) and np.all(c[:, 3] == ns) and np.all(n == len(c)) and len(c) <= 512
        assert np.array_equal(c[:, 2] & 0xffff, np.arange(len(c)))
        begin = s0 + np.arange(len(c)) * _span(ns)
        end = np.minimum(begin + _span(ns), s0 + ns)
        assert begin[0] == s0 and end[-1] == s0 + ns and np.all(end[:-1] == begin[1:]) and np.all(end > begin)
    assert len(chunk_list([])) == 0


def _eight_launch_iterations(b, inst, n_iter=8):
    """Iterations of the same system by mfv_krylov_tick, whose work arrays are made here."""
    import torch
    from manapy_amd import _lib
    from manapy_amd.device import stream_ptr
    w = _lib.MfvKrylovWork()
    R = b.S * 64
    x, scal, status = torch.zeros_like(b.x), b.scal.clone(), torch.zeros_like(b.status)
    part = torch.zeros(4 * b.S, dtype=torch.float64, device='cuda')
    vec = {k: torch.zeros(R, dtype=torch.float32, device='cuda') for k in ('d', 'r', 'rh', 'p', 'v', 'yz', 't', 'dinv')}
    status[inst] = _lib.KS_START
    w.x, w.b, w.partial, w.scal, w.status = (t.data_ptr() for t in (x, b.b, part, scal, status))
    for k, t in vec.items():
        setattr(w, k, t.data_ptr())
    gs, gi = b.grids()
    for _ in range(400):
        _lib.call('mfv_krylov_tick', b.eptr, ctypes.byref(w), n_iter, gs, gi, stream_ptr())
        if int(status[inst]) in (_lib.KS_DONE, _lib.KS_FAILED):
            break
    assert int(status[inst]) == _lib.KS_DONE
    return float(scal[inst * _lib.KS_NSCAL + _lib.KS_ITTOT])


# rows: under a slice, one slice, one chunk and one row more, ragged, and slices > 2048 (span 8)
@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("nx,ny,n_iter", [(2, 2, 8), (8, 4, 1), (16, 8, 3), (3, 43, 8), (37, 29, 8), (300, 230, 6)])
def test_solve_reaches_the_residual_in_as_many_iterations(nx, ny, n_iter):
    import torch
    from manapy_amd import _lib
    from manapy_amd.krylov import EllBatch
    d = make_tri_domain(nx, ny, 1.0, float(ny) / nx, 0.1, 5)
    C = int(d.nbcells)
    node_dir = torch.zeros(int(d.nbnodes), dtype=torch.uint8, device='cuda')
    rank = torch.full((int(d.nbfaces),), -1, dtype=torch.int32, device='cuda')
    b = EllBatch((C + 63) // 64 + 3, max_inst=2, width=32)
    b.alloc(100)  # the instance does not start at slice 0
    inst = b.alloc(C)
    b.publish()
    b.assemble_diamond(inst, d.device_diamond, node_dir, rank)
    rhs = torch.as_tensor(np.random.default_rng(nx).standard_normal(C), device='cuda')
    sigma, tau = 1.0, -2e-4 * nx / ny
    b.set_system(inst, sigma, tau, rhs)
    seen = [int(b.status[inst])]
    for _ in range(400):
        b.tick(n_iter)
        seen.append(int(b.status[inst]))
        if seen[-1] in (_lib.KS_DONE, _lib.KS_FAILED):
            break
    assert seen[-1] == _lib.KS_DONE, seen
    row0 = b.rows(inst)[0]
    x, y = b.x, torch.zeros_like(b.x)
    b.spmv(x, y)
    res = rhs - (sigma * x + tau * y)[row0:row0 + C]
    assert float(res.norm()) <= 1.0001e-10 * float(rhs.norm())  # the stop is 1e-10; 1e-4 for the other order of the sum
    mine = float(b.scalars(inst)[_lib.KS_ITTOT])
    b.scal[inst * _lib.KS_NSCAL + _lib.KS_ITTOT] = 0.
    ref = _eight_launch_iterations(b, inst)
    assert abs(mine - ref) <= 0.15 * ref + 3, (mine, ref)


# triangles between two Dirichlet sides, cells graded so that the diagonal varies by 2, 7e3, 1e2 and 1e4
@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("n,grade", [(12, 1.), (12, 100.), (30, 10.), (30, 100.)])
def test_graded_system_without_a_shift(n, grade):
    """sigma = 0 on a graded mesh, where the inner stop on the Jacobi-scaled residual is not the eight-launch
    solver's: the FP64 residual still meets the outer stop, in no more iterations."""
    import torch
    from manapy_amd import Domain, Variable, _lib, jittered_triangles
    from manapy_amd.solvers.ls import HIPKrylovSolver
    el, nd = jittered_triangles(n, n, 1., 1., .1, n)
    nd = nd.copy()
    if grade > 1.:
        nd[:, :2] = (grade ** nd[:, :2] - 1.) / (grade - 1.)
    d = Domain(2, mesh=(el, nd))
    var = Variable(domain=d, BC={"in": "dirichlet", "out": "dirichlet"}, values={"in": 1., "out": 2.})
    sol = HIPKrylovSolver(domain=d, var=var)
    C = int(d.nbcells)
    sol(rhs=np.random.default_rng(n).standard_normal(C))
    b, inst = sol._batch, sol._inst
    row0 = b.rows(inst)[0]
    y = torch.zeros_like(b.x)
    b.spmv(b.x, y)
    res = (b.b - y)[row0:row0 + C]
    assert float(res.norm()) <= 1.0001e-10 * float(b.b[row0:row0 + C].norm())
    for k in (_lib.KS_IT, _lib.KS_ITTOT, _lib.KS_OUTER):
        b.scal[inst * _lib.KS_NSCAL + k] = 0.
    ref = _eight_launch_iterations(b, inst, 64)  # up to 6000 iterations here
    assert sol.stats["iterations"] <= 1.15 * ref + 3, (sol.stats, ref)
