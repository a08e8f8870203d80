"""Batches captured into a graph of the caller's own: replays must not depend on
what the context runs in between, whatever it does to its workspace."""

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


@pytest.mark.parametrize("n,d", [(700, 2), (9000, 3), (60_000, 2)])
def test_replays_between_other_shapes(n, d):
    import torch
    db = _batch(n, d, 1).device(0)
    db.launch()
    want = db.results()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=db.stream):
        db.launch()
    assert db.stats()["knn_pairs"] >= 0
    # Shapes that move every buffer, and shapes that only use them (three: the
    # captured one stays among the four that are kept).
    others = [_batch(m, e, m) for m, e in ((200_000, 3), (300, 2), (400_000, 2))]
    ref = [b.run() for b in others]
    for turn in range(3):
        for b, r in zip(others, ref):
            db.out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(db.out.cpu().numpy(), want)
            np.testing.assert_array_equal(b.run(), r)
    # Eager runs of the captured shape use the shared workspace again.
    db.launch()
    np.testing.assert_array_equal(db.results(), want)
    db.out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(db.out.cpu().numpy(), want)


def test_new_shapes_are_not_captured():
    import torch
    old, new = _batch(500, 2, 2).device(0), _batch(501, 2, 2).device(0)
    old.launch()
    want = old.results()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=old.stream):
        old.launch()
        with pytest.raises(Exception, match="captured only after"):
            new.launch()
    old.out.zero_()
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(old.out.cpu().numpy(), want)
    new.launch()
    assert np.isfinite(new.results()).all()
