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


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("n,d", [(501, 2), (7000, 3), (60_001, 2)])
def test_new_shapes_are_captured(mode, n, d):
    """A shape's first run may be a recorded one: its tables are the graph's own,
    whatever tables and buffers go up for other shapes before a replay."""
    import torch
    old, new = _batch(500 + d, 2, 2).device(0), _batch(n, d, 3).device(0)
    old.launch()   # (queued on the stream when its capture begins)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=new.stream, capture_error_mode=mode):
        new.launch()
    others = [_batch(m + n, e, m) for m, e in ((100_000, 3), (300, 2))]
    ref = [b.run() for b in others]
    got = []
    for turn in range(2):
        for b, r in zip(others, ref):
            new.out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got.append(new.out.cpu().numpy())
            np.testing.assert_array_equal(b.run(), r)
    new.launch()   # the shape's first eager run
    want = new.results()
    assert np.isfinite(want).all()
    for g in got:
        np.testing.assert_array_equal(g, want)


def test_several_new_shapes_in_one_graph():
    import torch
    batches = [_batch(n, d, n).device(0) for n, d in ((450, 2), (2600, 3), (31_000, 2), (900, 4), (1200, 3), (5200, 2))]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=batches[0].stream):
        for b in batches:
            b.launch()
    for _ in range(3):
        for b in batches:
            b.out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = [b.out.cpu().numpy() for b in batches]
    for b, g in zip(batches, got):
        b.launch()
        np.testing.assert_array_equal(g, b.results())
