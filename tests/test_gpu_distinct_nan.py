"""NaN in discrete data: np.unique(axis=0) keeps every NaN a value of its own,
after +inf; the sorted distinct rows and the estimators on them must, too."""

import warnings

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


def _column(n, form, seed):
    rng = np.random.default_rng(seed)
    a = rng.integers(-2, 3, n) * 0.5
    pick = rng.random(n)
    if form in ("nan", "both"):
        a[pick < 0.3] = np.nan
    if form in ("inf", "both"):
        a[pick > 0.8] = np.inf
        a[(pick > 0.4) & (pick < 0.5)] = -np.inf
    if form == "only":
        a[:] = np.nan
    return a


SIZES = [1, 2, 3, 255, 1023, 1025, 2047, 2049, 8193, 16_384, 16_385, 20_000]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("form", ["nan", "inf", "both", "only"])
def test_one_column(n, form):
    from ennemi_amd import _discrete as d
    a = _column(n, form, n)
    rows, inverse, counts = np.unique(a, axis=0, return_inverse=True, return_counts=True)
    codes, got = d._device_unique([[a]])[0]
    np.testing.assert_array_equal(got, counts)
    np.testing.assert_array_equal(rows[codes], a)
    np.testing.assert_array_equal(np.bincount(codes, minlength=len(counts)), counts)
    # The numbers of the rows without NaN are np.unique's.
    whole = ~np.isnan(a)
    np.testing.assert_array_equal(codes[whole], np.ravel(inverse)[whole])


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("forms", [("nan", "inf"), ("both", "both"), ("inf", "nan", "both"), ("only", "inf")])
def test_rows(n, forms):
    from ennemi_amd import _discrete as d
    cols = [_column(n, f, n + 7 * i) for i, f in enumerate(forms)]
    table = np.column_stack(cols)
    _, inverse, counts = np.unique(table, axis=0, return_inverse=True, return_counts=True)
    # Several sets at once, of which some share columns.
    (codes, got), (_, first), (_, last) = d._device_unique([cols, cols[:1], [cols[-1]]])
    np.testing.assert_array_equal(got, counts)
    np.testing.assert_array_equal(np.bincount(codes, minlength=len(counts)), counts)
    whole = ~np.isnan(table).any(axis=1)
    np.testing.assert_array_equal(codes[whole], np.ravel(inverse)[whole])
    np.testing.assert_array_equal(first, np.unique(cols[0], axis=0, return_counts=True)[1])
    np.testing.assert_array_equal(last, np.unique(cols[-1], axis=0, return_counts=True)[1])


@pytest.mark.parametrize("n", [40, 3000])
def test_estimators_agree_with_oracle(n):
    import ennemi_amd
    a = _column(n, "both", n)
    table = np.column_stack([a, _column(n, "nan", n + 1)])
    rng = np.random.default_rng(n)
    x = rng.integers(0, 4, n) * 0.25
    y = (x + rng.integers(0, 2, n)) * 0.5
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        for v in (a, table):
            got = ennemi_amd.estimate_entropy(v, discrete=True, multidim=True)
            assert abs(got - orc.estimate_entropy(v, discrete=True, multidim=True)) <= 1e-12
            got = ennemi_amd.estimate_mi(y, x, cond=v, discrete_x=True, discrete_y=True)
            want = orc.estimate_mi(y, x, cond=v, discrete_x=True, discrete_y=True)
            np.testing.assert_allclose(got, want, rtol=0, atol=1e-12)
