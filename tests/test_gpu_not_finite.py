"""Rescaling a column that holds an infinity leaves no finite value in it: the
block, merge and sample sorts and the trees must then give the radii, counts and
values of the scan of all pairs, which passes NaN differences over.  (Two columns
of many points, which are cut into strips, are not among these: a strip's
neighbours are found by differences of the first column.)"""

import warnings

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,copies", [(64, 1), (300, 2), (2_000, 1), (2_049, 1), (9_000, 1), (20_000, 3), (50_000, 2)])
@pytest.mark.parametrize("dz", [0, 1, 2])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_against_all_pairs(n, copies, dz, which):
    import ennemi_amd
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    if which > 1 and dz == 0:
        which = 0
    rng = np.random.default_rng(n + dz)
    v = rng.normal(size=(n, 2 + dz))
    v[n // 2, which] = np.inf
    x, y, z = v[:, 0], v[:, 1], v[:, 2:] if dz else None
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        xs, ys, zs = orc.rescale_data(x, y, z, False, False)
        got = ennemi_amd.estimate_mi(y, x, cond=z)
    cols = [np.ascontiguousarray(c) for c in [xs, ys] + ([zs[:, c] for c in range(dz)] if dz else [])]
    assert np.isnan(cols[which]).all()

    def run(flags, copies):
        b = Batch()
        for _ in range(copies):
            c = [c.copy() for c in cols]
            b.add(nat.KIND_CMI if dz else nat.KIND_KSG, 3, c[:1], c[1:2], c[2:])
        return b.run(flags=flags, export=True)

    want, eps, counts = run(nat.F_BRUTE | nat.F_FP64, 1)
    for flags in (0, nat.F_FP64):
        values, e, c = run(flags, copies)
        for i in range(copies):
            np.testing.assert_array_equal(e[i], eps[0])
            np.testing.assert_array_equal(c[i], counts[0])
        np.testing.assert_allclose(values, want[0], rtol=0, atol=1e-12)
    np.testing.assert_allclose(got, [[want[0]]], rtol=0, atol=1e-12)


@pytest.mark.parametrize("n", [2, 511, 2_049, 8_193, 400_000, 900_000])
def test_one_column(n):
    """Keys of the sorted order: no neighbour at a finite distance, by any sort."""
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    a = np.full(n, np.nan)
    half = np.random.default_rng(n).normal(size=n)
    half[n // 2:] = np.nan
    b = Batch()
    b.add(nat.KIND_KL, 1, [a])
    b.add(nat.KIND_KL, 1, [half])
    b.add(nat.KIND_KL, 1, [half[:n // 2 + 1].copy()])
    _, (e, h, f), _ = b.run(export=True)
    assert np.isinf(e).all()
    s = np.sort(half[:n // 2])
    gap = np.concatenate([[np.inf], np.diff(s), [np.inf]])
    want = np.full(n, np.inf)
    want[np.argsort(half[:n // 2], kind="stable")] = np.minimum(gap[:-1], gap[1:])
    np.testing.assert_array_equal(h, want)
    np.testing.assert_array_equal(f, want[:n // 2 + 1])
