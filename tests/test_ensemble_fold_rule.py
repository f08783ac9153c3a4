"""The rule by which the steps of an ensemble graph fold the dt themselves, on the CPU: the partials that
all tiles read together, which one large instance among small ones drives far above what the mean
instance suggests."""
import ctypes

import numpy as np
import pytest

I32 = np.int32


def _rule(cells, tile=192):
    """(decision, bytes of partials, cells) for instances of ``cells`` triangles in tiles of ``tile``."""
    from manapy_amd import _lib
    n = np.asarray(cells, dtype=np.int64)
    waves = (n + 63) // 64
    cell0 = np.concatenate([[0], np.cumsum(waves * 64)[:-1]])
    inst = np.repeat(np.arange(len(n)), waves).astype(I32)
    tiles = np.concatenate([np.arange(c, c + w * 64, tile) for c, w in zip(cell0, waves)]).astype(I32)
    ncells, total = n.astype(I32), int(waves.sum()) * 64
    out = ctypes.c_int(-1)
    P = lambda a: a.ctypes.data
    _lib.call("mfv_sw_batch_fold_rule", total, len(n), P(ncells), len(inst), P(inst), len(tiles), P(tiles),
              ctypes.byref(out))
    reads = 8. * float(sum(-(-w * 64 // tile) * w for w in waves.tolist()))
    return out.value, reads, total


# both sides of the lines: 2100 tiles of 192 cells are 403k cells; 64 MB, 100 MB and 30 bytes a cell of partials
@pytest.mark.parametrize("cells,folds", [([8000] * 4, 1), ([3], 1), ([60000, 64], 1), ([390000], 1), ([400000], 0),
                                         ([200000] * 2, 1), ([22000] * 24, 1), ([60000] * 8, 0), ([1000] * 500, 1),
                                         ([600000] + [1000] * 23, 0)])
def test_decision(cells, folds):
    got, reads, total = _rule(cells)
    tiles = sum(-(-(-(-c // 64)) // 3) for c in cells)
    assert got == folds == int(reads <= 100e6 if tiles <= 2100 else reads <= 64e6 and reads <= 30. * total)


def test_one_large_instance_is_not_its_mean():
    """As many cells, tiles and instances: even sizes fold, one large instance does not."""
    even, uneven = [26000] * 24, [26000 * 24 - 23 * 1000] + [1000] * 23
    assert _rule(even)[0] == 1 and _rule(uneven)[0] == 0
    assert _rule(uneven)[1] > 20 * _rule(even)[1]


def test_bad_tables_are_refused():
    from manapy_amd import _lib
    a = np.zeros(2, dtype=I32)
    out = ctypes.c_int(0)
    for bad in (np.array([0, 128], I32), np.array([0, -64], I32)):
        with pytest.raises(_lib.MfvError, match="tile 1"):
            _lib.call("mfv_sw_batch_fold_rule", 128, 1, a.ctypes.data, 2, a.ctypes.data, 2, bad.ctypes.data,
                      ctypes.byref(out))
    with pytest.raises(_lib.MfvError, match="instance"):
        _lib.call("mfv_sw_batch_fold_rule", 64, 1, a.ctypes.data, 1, np.array([1], I32).ctypes.data, 1, a.ctypes.data,
                  ctypes.byref(out))
