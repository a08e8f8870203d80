"""The workspace that a context's plans share: runs of other shapes in
between move, grow and trim it, and captured graphs must follow."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(n, d, seed):
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    a = np.random.default_rng(seed).normal(size=(n, d))
    b = Batch()
    c = [np.ascontiguousarray(a[:, j]) for j in range(d)]
    b.add(nat.KIND_KSG, 3, c[:1], c[1:2])
    if d > 2:
        b.add(nat.KIND_CMI, 3, c[:1], c[1:2], c[2:])
        b.add(nat.KIND_KL, 4, c)
    return b


def test_graphs_and_plans_survive_other_shapes():
    import ennemi_amd._native as nat
    first = _batch(3000, 3, 1)
    graph = first.device(nat.F_GRAPH)
    eager = first.device(0)
    for db in (graph, eager):
        db.launch()
    ref = eager.results()
    np.testing.assert_array_equal(graph.results(), ref)
    # Larger, many, and much larger shapes, with replays in between.
    others = [_batch(n, d, n) for n, d in ((50_000, 2), (9000, 5), (300, 2), (400_000, 2), (64, 4), (5000, 3), (700, 3))]
    for turn in range(2):
        for b in others:
            db = b.device(0)
            db.launch()
            want = db.results()
            for db2 in (graph, eager):
                db2.launch()
            np.testing.assert_array_equal(graph.results(), ref)
            np.testing.assert_array_equal(eager.results(), ref)
            db.launch()
            np.testing.assert_array_equal(db.results(), want)
    assert graph.stats() is not None


def test_results_do_not_depend_on_what_ran_before():
    batches = [_batch(n, d, 10 * n) for n, d in ((2500, 3), (70_000, 2), (100, 3), (20_000, 4))]
    ref = [b.run() for b in batches]
    for order in ([3, 0, 1, 2], [2, 2, 3, 1, 0], [1, 0, 3, 2]):
        for i in order:
            np.testing.assert_array_equal(batches[i].run(), ref[i])
