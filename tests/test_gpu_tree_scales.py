"""Box trees of columns of unlike scales: the radii and counts of the scan of all
pairs, and no more points looked at than a few times those of like scales."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nat():
    import ennemi_amd._native as nat
    return nat


def _cols(n, d, scales, seed, form="plain"):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, d)) @ (np.eye(d) + 0.3)
    if form == "most equal":
        a[rng.random((n, d)) < 0.8] = 0.0
    elif form == "tails":
        a = rng.standard_t(1.2, size=(n, d))
    elif form == "constant":
        a[:, 0] = 1.0
    elif form == "infinite":
        a[rng.random(n) < 0.4, d - 1] = np.inf
    elif form == "all constant":
        a[:] = 2.0
    return [np.ascontiguousarray(a[:, c] * scales[c % len(scales)]) for c in range(d)]


@pytest.mark.parametrize("n", [64, 65, 128, 129, 1000, 4096, 4097, 20_011])
@pytest.mark.parametrize("d", [2, 3, 5, 9])
@pytest.mark.parametrize("form", ["plain", "most equal", "tails", "constant", "infinite", "all constant"])
def test_against_all_pairs(n, d, form):
    from ennemi_amd._batch import Batch
    nat = _nat()
    c = _cols(n, d, [1.0, 1e6, 1e-300 if form == "plain" else 1e-4, 30.0], n + d, form)
    b = Batch()
    b.add(nat.KIND_KL, 3, c)
    if d > 2:
        b.add(nat.KIND_CMI, 2, c[:1], c[1:2], c[2:])
        b.add(nat.KIND_ROSS, 2, c[1:], class_sizes=[n // 3, n - n // 3])
    _, eps, counts = b.run(nat.F_BRUTE | nat.F_FP64, export=True)
    _, e, k = b.run(0, export=True)
    for i in range(len(b)):
        np.testing.assert_array_equal(e[i], eps[i])
        np.testing.assert_array_equal(k[i], counts[i])


@pytest.mark.parametrize("d", [3, 4, 5])
@pytest.mark.parametrize("wide", [0, 1, 2])
def test_points_looked_at(d, wide):
    from ennemi_amd._batch import Batch
    nat = _nat()
    n = 100_000

    def looked_at(scales):
        b = Batch()
        b.add(nat.KIND_KL, 3, _cols(n, d, scales, d))
        db = b.device(0)
        db.launch()
        db.results()
        return db.stats()["knn_pairs"] / n

    like = looked_at([1.0])
    unlike = looked_at([1e6 if c == wide else 1.0 for c in range(d)])
    # At least the leaves of every cell that the wide column does not tell apart:
    # 25 cells, a leaf or two each.
    assert unlike <= max(2 * like, 3 * 64 * 25)
