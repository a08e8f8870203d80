"""Runs of one context on several streams, the default stream among them: a run
waits for the one before it, whose workspace it takes over."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(n, d, seed):
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    a = np.random.default_rng(seed).normal(size=(n, d))
    c = [np.ascontiguousarray(a[:, j]) for j in range(d)]
    b = Batch()
    b.add(nat.KIND_KSG, 3, c[:1], c[1:2])
    if d > 2:
        b.add(nat.KIND_CMI, 4, c[:1], c[1:2], c[2:])
    return b


def _launch(db, stream, static):
    db.stream = stream
    if static:
        db.ctx.run_static(db.inst_arr, db.n_inst, db.seg_arr, db.arena.data_ptr(), db.out.data_ptr(), 0, 0, 0,
                          stream.cuda_stream)
    else:
        db.launch()


@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("order", [("null", "a"), ("a", "null"), ("a", "b"), ("null", "a", "null", "b")])
def test_each_run_ends_before_the_next_begins(order, static):
    import torch
    streams = {"null": torch.cuda.default_stream(), "a": torch.cuda.Stream(), "b": torch.cuda.Stream()}
    assert streams["null"].cuda_stream == 0
    # Long runs first, short ones of other shapes after them.
    shapes = [(150_000, 3), (400, 2), (20_000, 3), (3000, 2)]
    dbs = [_batch(n, d, n).device(0) for n, d in shapes]
    ref = []
    for db in dbs:
        db.launch()
        ref.append(db.results())
    for first in range(len(dbs)):
        torch.cuda.synchronize()
        turn = [(dbs[(first + i) % len(dbs)], ref[(first + i) % len(dbs)]) for i in range(len(order))]
        for db, _ in turn:
            db.out.zero_()
        torch.cuda.synchronize()
        for name, (db, _) in zip(order, turn):
            _launch(db, streams[name], static)
        torch.cuda.synchronize()
        for db, want in turn:
            np.testing.assert_array_equal(db.out.cpu().numpy(), want)
