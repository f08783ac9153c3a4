"""Mesh tables as a caller of the C ABI may hold them: what the residual orders hold past a cell's face
count, and where the tables begin, changes nothing."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available
from test_gpu_mixed_meshes import tri_quad_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _descriptor(m, **tables):
    """A copy of the mesh's descriptor with some tables replaced."""
    from manapy_amd import _lib
    d = _lib.MfvMesh()
    ctypes.memmove(ctypes.byref(d), ctypes.byref(m.desc), ctypes.sizeof(d))
    for k, t in tables.items():
        setattr(d, k, t.data_ptr())
    return d


def _results(m, desc, order):
    """Residuals, time step and a fused step of random fields through the ABI."""
    import torch
    from manapy_amd import _lib
    from manapy_amd.device import stream_ptr
    g = torch.Generator(device="cuda").manual_seed(3)
    C, F = int(m.C), int(m.F)
    cell = [torch.randn(C, dtype=torch.float64, device="cuda", generator=g) for _ in range(8)]
    face = [torch.randn(F, dtype=torch.float64, device="cuda", generator=g) for _ in range(4)]
    rez, dis, out = (torch.zeros(C, dtype=torch.float64, device="cuda") for _ in range(3))
    dt = torch.zeros(1, dtype=torch.float64, device="cuda")
    ring = torch.zeros(4, dtype=torch.float64, device="cuda")
    scratch = torch.zeros(4 * C, dtype=torch.float64, device="cuda")
    p, s, ptr = ctypes.byref(desc), stream_ptr(), lambda ts: [t.data_ptr() for t in ts]
    _lib.call("mfv_explicitscheme_convective", p, rez.data_ptr(), cell[0].data_ptr(), *ptr(face), *ptr(cell[1:5]),
              order, s)
    _lib.call("mfv_explicitscheme_dissipative", p, *ptr(face[:2]), None, .1, .2, 0., dis.data_ptr(), s)
    _lib.call("mfv_time_step", p, *ptr(cell[5:8]), .4, dt.data_ptr(), None, s)
    _lib.call("mfv_dt_ring_init", ring.data_ptr(), dt.data_ptr(), s)
    _lib.call("mfv_advection_step", p, cell[0].data_ptr(), out.data_ptr(), *ptr(cell[5:8]), *ptr(face[1:4]), .4,
              order, ring.data_ptr(), 0, scratch.data_ptr(), s)
    return [rez, dis, dt, ring, out]


def _equal(a, b):
    import torch
    assert all(torch.equal(x, y) for x, y in zip(a, b))


# triangles (three of four slots used) beside quadrilaterals; 63 cells: less than a wave
@pytest.mark.parametrize("size", [(7, 5), (31, 23)])
@pytest.mark.parametrize("order", [1, 2])
def test_order_rows_past_the_face_count(size, order):
    """The order tables' rows past a cell's count may hold anything."""
    import torch
    d = tri_quad_domain(*size, 100., 70.)
    m = d.device_mesh
    m.ensure_lsq()
    want = _results(m, m.desc, order)
    past = torch.arange(m.MF, device="cuda")[:, None] >= m.t["cell_nfaces"][None, :]
    assert bool(past.any())
    filled = {}
    for k in ("order_split", "order_sorted"):
        t = m.t[k].clone()
        t[past] = 255
        filled[k] = t
    _equal(_results(m, _descriptor(m, **filled), order), want)


@pytest.mark.parametrize("order", [1, 2])
def test_face_cells_aligned_to_four_bytes(order):
    """face_cells is an int32 table: its first entry may lie at any multiple of 4."""
    import torch
    d = tri_quad_domain(31, 23, 100., 70.)
    m = d.device_mesh
    m.ensure_lsq()
    want = _results(m, m.desc, order)
    n = 2 * int(m.F)
    odd = torch.empty(n + 1, dtype=torch.int32, device="cuda")[1:]
    odd.copy_(m.t["face_cells"].reshape(-1))
    assert odd.data_ptr() % 8 == 4
    _equal(_results(m, _descriptor(m, face_cells=odd), order), want)
