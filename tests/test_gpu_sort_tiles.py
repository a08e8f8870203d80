"""First-stage sorts at the edges of their tiles (512 to 8,192 keys), merge
passes and the change to the sample sort (750,000 keys), and the packing of its
buckets; keys of every kind, and columns that hold no finite value."""

import warnings

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _keys(n, form, rng):
    a = rng.normal(size=n)
    if form == "ties":
        return np.round(a, 1)
    if form == "equal":
        return np.full(n, 0.5)
    if form == "skewed":   # buckets of very different sizes
        return np.where(rng.random(n) < 0.7, rng.integers(0, 3, n).astype(float), a * 1e3)
    if form == "falling":
        return -np.sort(a)
    return a


def _nearest(a):
    """Distance of every point to its nearest other one."""
    order = np.argsort(a, kind="stable")
    s = a[order]
    gap = np.concatenate([[np.inf], np.diff(s), [np.inf]])
    d = np.empty(len(a))
    d[order] = np.minimum(gap[:-1], gap[1:])
    return d


@pytest.mark.parametrize("form", ["normal", "ties", "equal", "skewed", "falling"])
@pytest.mark.parametrize("sizes", [(2,), (511, 512), (513, 1024), (1025, 2048), (2049,), (4096, 3), (4097,), (8192, 8191),
                                   (8193, 2048, 1), (16_384, 16_385), (40_000,), (375_000, 375_000), (375_001, 375_000),
                                   (5_000,) * 151, (900_000, 17), (1_100_000,)])
def test_one_column_sorts(sizes, form):
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    rng = np.random.default_rng(len(sizes) + sizes[0])
    cols = [_keys(n, form, rng) for n in sizes]
    b = Batch()
    for c in cols:
        if len(c) > 1:
            b.add(nat.KIND_KL, 1, [c])
    _, eps, _ = b.run(export=True)
    for c, e in zip([c for c in cols if len(c) > 1], eps):
        np.testing.assert_array_equal(e, _nearest(c))


@pytest.mark.parametrize("n", [300, 2_000, 2_049, 9_000, 20_000])
@pytest.mark.parametrize("dz", [0, 1])
def test_columns_without_finite_values(n, dz):
    # Rescaling a column that holds an infinity leaves no finite value.
    import ennemi_amd
    rng = np.random.default_rng(n)
    y, x = rng.normal(size=(2, n))
    x[n // 2] = np.inf
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        out = ennemi_amd.estimate_mi(y, x, k=3, cond=rng.normal(size=n) if dz else None)
    assert out.shape == (1, 1)
