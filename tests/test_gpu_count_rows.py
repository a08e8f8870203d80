"""Distinct rows counted directly (whole numbers in small ranges) and by
sorting: both ways must give np.unique's rows and counts, at the edges of the
counters (in LDS up to 8,192 keys, at most 65,536), of the row sets that one
workgroup counts (16,384) and of the sort tiles."""

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


def _rows(n, radix, seed, kind=np.int64):
    rng = np.random.default_rng(seed)
    cols = [rng.integers(0, r, size=n) - r // 2 for r in radix]
    for c, r in zip(cols, radix):
        c[:1] = -(r // 2)
        c[-1:] = r - 1 - r // 2
    return [c.astype(kind) for c in cols]


def _check(cols):
    from ennemi_amd import _discrete as d
    got = d._count_rows(cols)
    rows, counts = np.unique(np.column_stack([c.astype(np.float64) for c in cols]), axis=0, return_counts=True)
    if got is not None:
        codes, c, _ = got
        np.testing.assert_array_equal(c, counts)
        for j, col in enumerate(cols):
            np.testing.assert_array_equal(codes[j] + float(col.min()), rows[:, j])
    codes, c = d._device_unique([cols])[0]
    np.testing.assert_array_equal(c, counts)
    np.testing.assert_array_equal(rows[codes], np.column_stack(cols))
    return got is not None


@pytest.mark.parametrize("n", [1, 2, 255, 1023, 1025, 2047, 2048, 2049, 16_384, 16_385, 40_001])
@pytest.mark.parametrize("radix,direct", [((1,), True), ((2, 3), True), ((64, 128), True), ((64, 129), True),
                                          ((256, 256), True), ((256, 257), False), ((4, 5, 6, 7), True)])
def test_ranges(n, radix, direct):
    if n == 1:
        radix, direct = (1,) * len(radix), True
    assert _check(_rows(n, radix, n)) == direct


@pytest.mark.parametrize("kind", [np.int8, np.int16, np.int32, np.float32, np.float64])
def test_types(kind):
    assert _check(_rows(3000, (9, 5), 4, kind))
    assert _check([c > 1 for c in _rows(3000, (9, 5), 4)])


def test_values_that_are_sorted_instead():
    x = np.random.default_rng(1).integers(0, 7, 5000).astype(float)
    assert not _check([x + 0.5])
    assert not _check([x * 1e6])
    assert not _check([np.where(x == 3, 2.0 ** 60, x)])
    assert _check([x + 2.0 ** 52])
    x[::3] = -0.0
    assert _check([x])


@pytest.mark.parametrize("scale", [1.0, 0.25, 1e7])
def test_estimators_agree_with_oracle(scale):
    """The same labels as small whole numbers, fractions and far apart."""
    import warnings

    from ennemi_amd import _discrete as d
    rng = np.random.default_rng(2)
    n = 9000
    z = rng.integers(0, 3, size=(n, 2)) * scale
    x = rng.integers(-4, 5, size=n) * scale
    y = (np.abs(x) + z[:, 0]) * scale
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        assert d.estimate_discrete_mi(x, y) == orc.estimate_discrete_mi(x, y)
        assert d.estimate_conditional_discrete_mi(x, y, z) == orc.estimate_conditional_discrete_mi(x, y, z)
        assert abs(d.estimate_discrete_entropy(z) - orc.estimate_discrete_entropy(z)) <= 1e-12
