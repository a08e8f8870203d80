"""One-column kNN (windows of the sorted keys): radii against the oracle at
scope ends, item edges (2,048 positions), k from 1 to beyond the scope, ties,
and classes; infinities leave no neighbour among equals."""

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


def _nat():
    import ennemi_amd._native as nat
    return nat


@pytest.mark.parametrize("form", ["plain", "ties", "equal"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 257, 2047, 2048, 2049, 5000])
def test_entropy_radii(n, form):
    from ennemi_amd._batch import Batch
    nat = _nat()
    x = np.random.default_rng(n).normal(size=n)
    if form == "ties":
        x = np.round(x, 1)
    elif form == "equal":
        x[:] = 0.5
    ks = [1, 2, 3, 4, 7, 31, 100, 1000, n - 1, n, 3 * n]
    b = Batch()
    for k in ks:
        b.add(nat.KIND_KL, max(k, 1), [x])
    _, eps, _ = b.run(export=True)
    d = np.sort(np.abs(x[:, None] - x[None, :]), axis=1)
    for k, e in zip(ks, eps):
        k = max(k, 1)
        np.testing.assert_array_equal(e, d[:, k] if k < n else np.full(n, np.inf), err_msg=f"k={k}")


@pytest.mark.parametrize("k", [1, 3, 40])
def test_ross_classes(k):
    from ennemi_amd._batch import Batch
    nat = _nat()
    sizes = [1, 40, 41, 42, 2500, 3000]
    n = sum(sizes)
    rng = np.random.default_rng(k)
    x = np.round(rng.normal(size=n), 3)
    b = Batch()
    b.add(nat.KIND_ROSS, k, [x], class_sizes=sizes)
    b.add(nat.KIND_ROSS, k, [x], class_sizes=[n])
    vals, eps, cnts = b.run(export=True)
    for i, y in enumerate((np.repeat(np.arange(len(sizes)), sizes), np.zeros(n, dtype=int))):
        w, ref = orc.estimate_semidiscrete_mi(x, y, k, detail=True)
        np.testing.assert_array_equal(eps[i], ref["eps"])
        np.testing.assert_array_equal(cnts[i][0], ref["n_full"])
        assert vals[i] == w or abs(vals[i] - w) <= 1e-12


def test_infinities():
    from ennemi_amd._batch import Batch
    nat = _nat()
    x = np.random.default_rng(3).normal(size=500)
    x[[3, 77, 400]] = np.inf
    x[[9, 10]] = -np.inf
    b = Batch()
    b.add(nat.KIND_KL, 2, [x])
    _, eps, _ = b.run(export=True)
    fin = np.isfinite(x)
    d = np.sort(np.abs(x[fin][:, None] - x[fin][None, :]), axis=1)
    np.testing.assert_array_equal(eps[0][fin], d[:, 2])
    assert np.all(np.isinf(eps[0][~fin]))
