"""Ensemble graphs whose steps fold the dt themselves against the eager steps (a fold launch each):
states and dt rings bit for bit, over several replays with eager work between them; instances from a
part of a wave to more partials than a block has threads."""
import numpy as np
import pytest

from conftest import gpu_available, make_tri_domain

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("sizes", [[(3, 2)], [(3, 2), (11, 7), (16, 8)], [(150, 130), (3, 2), (40, 31)]])
@pytest.mark.parametrize("config", [("staged", 256, 256), ("staged", 128, 64), ("tiled", 256, 192)])
def test_graph_equals_eager(sizes, config):
    import torch
    from manapy_amd.ensemble import SwEnsemble
    doms, states = [], []
    for k, (nx, ny) in enumerate(sizes):
        d = make_tri_domain(nx, ny, 10., 10. * ny / nx, seed=k)
        rng = np.random.default_rng(k)
        C = int(d.nbcells)
        doms.append(d)
        states.append((1. + rng.random(C), .1 * rng.normal(size=C), .1 * rng.normal(size=C), .1 * rng.random(C)))
    a, b = SwEnsemble(doms, states), SwEnsemble(doms, states)
    for chunk in (6, 6, 12):
        a.run_graph(chunk, chunk=chunk, config=config)
        b.step(chunk, config=config)
        torch.cuda.synchronize()
        assert torch.equal(a.state, b.state)
        assert torch.equal(a.rings, b.rings)
        a.rings[:, 3] += 0.  # eager work of the caller's between replays


def test_graph_with_a_fold_launch_a_step():
    """More than 2100 tiles whose instance is large: the rule (mfv_sw_batch_fold_rule) leaves the dt to a launch."""
    test_graph_equals_eager([(300, 240), (3, 2)], ("staged", 128, 64))
