"""mfv_ghost_values: every boundary kind, more segments than one launch holds, and arrays that
are exchanged between calls, against the per-location definition (bit for bit)."""
import numpy as np
import pytest

from conftest import gpu_available, make_tet_domain, make_tri_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

KINDS = ["neumann", "dirichlet", "nonslip", "neumannNH", "slip", "dirichlet"]


def _expected(d, var, before):
    g = before.copy()
    own = d.faces.cellid[:, 0]
    w = var.cell.cpu().numpy()
    for bc in var.BCs.values():
        f = bc.BCfaces
        if bc.BCtype == "dirichlet":
            g[f] = bc.BCvalueface.cpu().numpy()[f]
        elif bc.BCtype == "neumannNH":
            g[f] = w[own[f]] + bc.constNH.cpu().numpy()[f] * d.faces.dist_ortho[f]
        else:
            g[f] = -w[own[f]] if bc.BCtype == "nonslip" else w[own[f]]
    return g


@pytest.mark.parametrize("dim,nvar", [(2, 1), (2, 9), (3, 1), (3, 6)])  # 4 to 36 segments (32 a launch)
def test_ghosts_of_all_kinds(dim, nvar):
    import torch
    from manapy_amd import Variable
    from manapy_amd.variable import fill_ghosts
    d = make_tri_domain(17, 5) if dim == 2 else make_tet_domain(4)
    rng = np.random.default_rng(dim + nvar)
    locs = ["in", "out", "bottom", "upper"] + (["front", "back"] if dim == 3 else [])
    vs = []
    for k in range(nvar):
        kinds = KINDS if dim == 2 else [t for t in KINDS if t != "neumannNH"]  # its distances are 2D
        bc = {loc: kinds[(k + i) % len(kinds)] for i, loc in enumerate(locs)}
        v = Variable(domain=d, BC=bc, values={loc: float(rng.normal()) for loc in locs})
        v.cell[:] = torch.as_tensor(rng.normal(size=int(d.nbcells)))
        v.ghost[:] = torch.as_tensor(rng.normal(size=int(d.nbfaces)))
        vs.append(v)
    cache = []
    for _ in range(3):
        want = [_expected(d, v, v.ghost.cpu().numpy()) for v in vs]
        fill_ghosts(d, [(b, v) for v in vs for b in v.BCs.values()], cache)
        for v, w in zip(vs, want):
            assert np.array_equal(v.ghost.cpu().numpy(), w)
        # other arrays under the same variable, other values in the same arrays
        vs[0].cell = torch.as_tensor(rng.normal(size=int(d.nbcells)), device='cuda')
        vs[-1].cell.mul_(1.5)
    v = vs[0]
    v.ghost.fill_(7.)
    want = _expected(d, v, v.ghost.cpu().numpy())
    v.update_ghost_value()
    assert np.array_equal(v.ghost.cpu().numpy(), want)
