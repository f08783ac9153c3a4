"""Stencil tiles of tetrahedral meshes: the host tables list every stencil in its order (CPU), and the
tiled gradient gives the bits of the gathering one (a part of a wave, several tiles with a remainder,
every kind of boundary value)."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available, make_tet_domain


@pytest.mark.parametrize("n,T", [(2, 256), (3, 64), (5, 256)])
def test_tables_hold_every_stencil(n, T):
    from manapy_amd import _lib
    from manapy_amd.device import gpu_layout
    from manapy_amd.renumber import morton_order_3d
    H = gpu_layout(make_tet_domain(n), lsq=True)
    C, K = H["C"], H["K"]
    perm = np.ascontiguousarray(morton_order_3d(*H["cell_center"].T), dtype=np.int64)
    h = _lib.MfvStencilTilesHost()
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    _lib.call("mfv_stencil_tiles_build", C, K, P(H["lsq_cells"]), P(H["lsq_ncells"]), P(perm), T, ctypes.byref(h))
    take = lambda p, m: np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_int32)), (m,)).copy()  # noqa: E731
    N = h.nb_tiles * T
    cell, eptr = take(h.cell, N), take(h.ext_ptr, h.nb_tiles + 1)
    ext, pairs = take(h.ext_cells, h.ext_len), take(h.pairs, h.nb_pairs * N).view(np.uint32).reshape(h.nb_pairs, N)
    max_ext = h.max_ext
    _lib.call("mfv_stencil_tiles_host_free", ctypes.byref(h))
    assert np.array_equal(cell[:C], perm) and np.all(cell[C:] == -1)
    most = 0
    for t in range(len(eptr) - 1):
        e = ext[eptr[t]:eptr[t + 1]]
        most = max(most, len(e))
        assert np.all(np.diff(e) > 0)
        for q in range(t * T, min((t + 1) * T, C)):
            nn = H["lsq_ncells"][cell[q]]
            pos = [(pairs[k // 2, q] >> (16 * (k % 2))) & 0xffff for k in range(nn)]
            assert np.array_equal(e[pos], H["lsq_cells"][:nn, cell[q]])
    assert most == max_ext


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("n", [2, 5, 9])
def test_tiled_gradient_equals_the_gathering_one(n):
    import torch
    from manapy_amd import Variable, _lib
    from manapy_amd.device import stream_ptr
    d = make_tet_domain(n)
    rng = np.random.default_rng(n)
    kinds = ("dirichlet", "neumann", "nonslip", "neumann", "dirichlet", "slip")
    v = Variable(domain=d, BC=dict(zip(("in", "out", "bottom", "upper", "front", "back"), kinds)),
                 values={"in": .3, "front": -1.})
    v.cell[:] = torch.as_tensor(rng.normal(size=int(d.nbcells)), device="cuda")
    v.update_ghost_value()
    m = d.device_mesh
    assert m.stencil_tiles() is not None
    v.compute_cell_gradient()
    got = [x.clone() for x in (v.gradcellx, v.gradcelly, v.gradcellz, v.psi)]
    f = (_lib.MfvGradientFields * 1)((v.cell.data_ptr(), v.ghost.data_ptr(), v.gradcellx.data_ptr(),
                                      v.gradcelly.data_ptr(), v.gradcellz.data_ptr(), v.psi.data_ptr()))
    for x in (v.gradcellx, v.gradcelly, v.gradcellz, v.psi):
        x.fill_(np.nan)
    _lib.call("mfv_cell_gradient_limited", m.ptr, 1, f, stream_ptr())
    for a, b in zip(got, (v.gradcellx, v.gradcelly, v.gradcellz, v.psi)):
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


def test_stencils_too_wide_for_a_tile_are_gathered(monkeypatch):
    """A tile that reads more cells than its 16-bit positions tell apart: the builder refuses it and the
    mesh has no tiles, so that its gradients gather from memory as without them."""
    from types import SimpleNamespace
    import torch
    from manapy_amd import _lib
    from manapy_amd.device import DeviceMesh, StencilTiles
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)  # asks for a device
    C, K = 66600, 260
    cells = np.zeros((K, C), dtype=np.int32)
    cells[:, :256] = np.arange(256 * K, dtype=np.int32).reshape(K, 256)
    count = np.where(np.arange(C) < 256, K, 0).astype(np.int32)
    x = np.linspace(0., 1., C)
    host = {"C": C, "K": K, "lsq_cells": cells, "lsq_ncells": count, "cell_center": np.stack([x, x, x], axis=1)}
    with pytest.raises(_lib.MfvError, match="65535"):
        StencilTiles(host, np.arange(C), "cpu")
    mesh = SimpleNamespace(ensure_lsq=lambda: None, _stencil_tiles=None, _lsq_host=None, host=host, dim=3, MF=4, C=C,
                           device="cpu")
    assert DeviceMesh.stencil_tiles(mesh) is None
    assert DeviceMesh.stencil_tiles(mesh) is None  # and does not build them again
    assert mesh._stencil_tiles is False


def test_a_failed_allocation_is_an_error_code():
    """A table larger than the address space: the entry point answers with a code, no exception leaves it."""
    from manapy_amd import _lib
    h = _lib.MfvStencilTilesHost()
    one, perm = np.zeros(1, dtype=np.int32), np.zeros(1, dtype=np.int64)
    with pytest.raises(_lib.MfvError, match="allocation failed"):
        _lib.call("mfv_stencil_tiles_build", 1, 2 ** 31 - 2, one.ctypes.data, one.ctypes.data, perm.ctypes.data, 1 << 20,
                  ctypes.byref(h))
    assert not h.pairs and not h.cell
