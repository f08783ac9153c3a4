"""What a request is charged against the HBM budget is what the arena holds for it."""
import pytest

from conftest import gpu_available, make_tri_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _tensor_bytes(arena):
    """Bytes of every distinct device tensor that the arena holds (views of another one left out)."""
    import torch
    seen = {}

    def take(v):
        if isinstance(v, torch.Tensor):
            if v._base is None:
                seen[v.data_ptr()] = v.numel() * v.element_size()
        elif isinstance(v, dict):
            [take(x) for x in v.values()]
    [take(v) for v in vars(arena).values()]
    return sum(seen.values())


@pytest.mark.parametrize("width", [1, 16, 32])
@pytest.mark.parametrize("slots", [0, 4, 8])
def test_bytes_per_slice_is_what_a_slice_adds(width, slots):
    from manapy_amd.krylov import EllBatch
    sizes = []
    for S in (64, 128):
        b = EllBatch(S, max_inst=3, width=width)
        if slots:
            b.enable_advection(slots)
        sizes.append((_tensor_bytes(b), b.bytes_per_slice()))
    assert sizes[0][1] == sizes[1][1] == (sizes[1][0] - sizes[0][0]) / 64


def test_an_admitted_request_holds_its_footprint():
    """Nothing but the arena's rows stays on the device after admission."""
    import numpy as np
    import torch
    from manapy_amd.serving import AdvDiffRequest, ServingEngine
    eng = ServingEngine(max_cells=1 << 13, max_inst=4)
    d = make_tri_domain(41, 37, 1., 1., .1, 3)
    r = AdvDiffRequest(0, d, np.ones(int(d.nbcells)), nsteps=2).prepare()
    eng.admit(AdvDiffRequest(1, d, np.ones(int(d.nbcells)), nsteps=2).prepare(), 0.)  # pools, first launches
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    eng.admit(r, 0.)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() - before == 0
    assert eng.in_use == 2 * r.footprint(eng.arena) == 2 * -(-int(d.nbcells) // 64) * eng.arena.bytes_per_slice()
