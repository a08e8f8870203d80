"""The instance tables of batches of device-prepared columns."""

import ctypes

import numpy as np

import ennemi_amd._native as nat


def _same(batch, inst_arr):
    for t, inst in zip(batch._inst, inst_arr):
        kind, k, n, dx, dy, dz, n_segs, seg_index, cols = t
        assert (inst.kind, inst.k, inst.n, inst.dx, inst.dy, inst.dz) == (kind, k, n, dx, dy, dz)
        assert (inst.n_segs, inst.seg_index) == (n_segs, seg_index)
        assert list(inst.col[:len(cols)]) == cols


def test_instances_of_classes():
    from ennemi_amd._batch import ArenaBatch
    b = ArenaBatch(None)
    b.add_many(nat.KIND_CROSS, 3, [7, 5, 9], [[0, 7], [14, 19], [24, 33]], 1, 0, 1)
    b.set_classes(np.array([[3, 0, 4], [5, 0, 0], [2, 3, 4]]))
    inst_arr, seg_arr = b.pack()
    _same(b, inst_arr)
    assert [(t[6], t[7]) for t in b._inst] == [(2, 0), (1, 2), (3, 3)]
    assert list(seg_arr) == [3, 4, 5, 2, 3, 4]
    assert isinstance(seg_arr, ctypes.Array)


def test_instances_without_classes():
    from ennemi_amd._batch import ArenaBatch
    b = ArenaBatch(None)
    b.add_many(nat.KIND_KSG, 3, [7, 5], [[0, 7], [14, 19]], 1, 1, 0)
    b.add(nat.KIND_CMI, 4, 6, [24, 30, 36], 1, 1, 1)
    _same(b, b.pack()[0])
    assert len(b._inst) == len(b) == 3
