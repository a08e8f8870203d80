"""Batches whose box trees do not fit the static workspace run on the sorted
orders alone, also where a strip size above those that LDS holds is set."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strip", [0, 2048, 65_536])
@pytest.mark.parametrize("kind,n", [("ROSS", 3_000_000), ("CROSS", 2_600_000)])
def test_two_columns_in_one_class(kind, n, strip):
    import torch

    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    rng = np.random.default_rng(n)
    x, z = rng.random((2, n))
    b = Batch()
    if kind == "ROSS":
        b.add(nat.KIND_ROSS, 3, [x, z], class_sizes=[n])
    else:
        b.add(nat.KIND_CROSS, 3, [x], z=[z], class_sizes=[n])
    db = b.device(0, export=True)
    db.launch()
    value, eps, counts = db.results()
    db.eps.fill_(-1.0)
    db.counts.fill_(-1)
    db.out.fill_(-1.0)
    torch.cuda.synchronize()
    old = db.ctx.get_tuning()
    try:
        db.ctx.set_tuning(strip, old[1])
        with db.ctx.lock:
            db.ctx.run_static(db.inst_arr, db.n_inst, db.seg_arr, db.arena.data_ptr(), db.out.data_ptr(),
                              db.eps.data_ptr(), db.counts.data_ptr(), db.flags, db.stream.cuda_stream)
        db.stream.synchronize()
        # (Trees would be cut from slabs, a second sort of every point.)
        assert db.stats()["sort_keys"] == n
        value2, eps2, counts2 = db.results()
        np.testing.assert_array_equal(value2, value)
        np.testing.assert_array_equal(eps2[0], eps[0])
        np.testing.assert_array_equal(counts2[0], counts[0])
    finally:
        db.ctx.set_tuning(*old)
