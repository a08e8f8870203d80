"""Box trees: radii and counts of spaces of two or more columns.

Sizes at the edges of leaves (64), cells (4,096), the slabs that longer
scopes are cut from (more than four cells) and groups of cells (more than 64),
every column class and both list lengths, against the oracle; every form also
against the plain key-order kernels (tuned without strips), which must give
the same bits.
"""

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


def _nat():
    import ennemi_amd._native as nat
    return nat


def _cols(a):
    return [np.ascontiguousarray(a[:, c]) for c in range(a.shape[1])]


def _data(n, d, seed, form="plain"):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, d)) @ rng.normal(size=(d, d))
    if form == "ties":
        a = np.round(a, 1)
    elif form == "tails":
        a = rng.standard_t(1.5, size=(n, d))
    elif form == "equal":
        a[:, 1:] = 0.25
    elif form == "infinite":
        a[rng.integers(0, n, 5), d - 1] = np.inf
        a[rng.integers(0, n, 5), d - 1] = -np.inf
    return a


def _both(build):
    """(values, radii, counts) by trees, checked bit for bit against the plain kernels."""
    nat = _nat()
    from ennemi_amd._batch import Batch
    ctx = nat.context()
    old = ctx.get_tuning()
    got = []
    try:
        for strip in (1024, 0):
            ctx.set_tuning(strip, old[1])
            b = Batch()
            build(b)
            got.append(b.run(export=True))
    finally:
        ctx.set_tuning(*old)
    np.testing.assert_array_equal(got[0][0], got[1][0])
    for which in (1, 2):
        for t, p in zip(got[0][which], got[1][which]):
            np.testing.assert_array_equal(t, p)
    return got[0]


SIZES = [2, 63, 64, 65, 128, 129, 1025, 2049, 4095, 4096, 4097, 12289, 16385]


@pytest.mark.parametrize("form", ["plain", "ties", "tails", "equal"])
@pytest.mark.parametrize("n", SIZES)
def test_sizes_and_forms(n, form):
    """Entropy of three columns and conditional MI with one and two
    conditions in one batch."""
    nat = _nat()
    k = min(3, n - 1)
    a = _data(n, 5, n, form)

    def build(b):
        b.add(nat.KIND_KL, k, _cols(a[:, :3]))
        b.add(nat.KIND_CMI, k, _cols(a[:, :1]), _cols(a[:, 1:2]), _cols(a[:, 2:3]))
        b.add(nat.KIND_CMI, k, _cols(a[:, :1]), _cols(a[:, 1:2]), _cols(a[:, 2:4]))

    vals, eps, cnts = _both(build)
    w, ref = orc.estimate_single_entropy(a[:, :3], k, detail=True)
    np.testing.assert_array_equal(eps[0], ref["eps"])
    for i, dz in ((1, 1), (2, 2)):
        w, ref = orc.estimate_conditional_mi(a[:, :1], a[:, 1:2], a[:, 2:2 + dz], k, detail=True)
        np.testing.assert_array_equal(eps[i], ref["eps"])
        for s, key in enumerate(("nxz", "nyz", "nz")):
            np.testing.assert_array_equal(cnts[i][s], ref[key], err_msg=key)
        assert vals[i] == w or abs(vals[i] - w) <= 1e-12 or (np.isnan(w) and np.isnan(vals[i]))


@pytest.mark.parametrize("form", ["plain", "ties"])
@pytest.mark.parametrize("k", [255, 256, 511, 512, 1100, 1999, 2000])
@pytest.mark.parametrize("d", [2, 3, 16])
def test_long_lists(d, k, form):
    """The longest lists, and those that take several passes (ties at the
    rank where one ends), up to more neighbours than points."""
    nat = _nat()
    a = _data(2000, d, 7 * d + k, form)
    _, eps, _ = _both(lambda b: b.add(nat.KIND_KL, k, _cols(a)))
    _, ref = orc.estimate_single_entropy(a, k, detail=True)
    np.testing.assert_array_equal(eps[0], ref["eps"])


@pytest.mark.parametrize("k", [3, 63, 64, 127, 128])
@pytest.mark.parametrize("d", [2, 3, 4, 5, 6, 7, 9, 13, 16])
def test_columns_and_list_lengths(d, k):
    """Every column class and the ends of the shorter list lengths (two
    columns with short lists run on strips)."""
    nat = _nat()
    a = _data(5000, d, 31 * d + k)
    _, eps, _ = _both(lambda b: b.add(nat.KIND_KL, k, _cols(a)))
    _, ref = orc.estimate_single_entropy(a, k, detail=True)
    np.testing.assert_array_equal(eps[0], ref["eps"])


@pytest.mark.parametrize("sizes", [[1, 2, 61], [64, 1, 4097], [4096, 4096, 9000], [20_000, 70, 3]])
@pytest.mark.parametrize("k", [4, 100])
def test_classes(sizes, k):
    """Trees of every class (Ross and its conditional form), some with fewer
    points than neighbours, and of all points together."""
    nat = _nat()
    n = sum(sizes)
    a = _data(n, 4, n + k)
    vals, eps, cnts = _both(lambda b: (b.add(nat.KIND_ROSS, k, _cols(a[:, :2]), class_sizes=sizes),
                                       b.add(nat.KIND_CROSS, k, _cols(a[:, :1]), z=_cols(a[:, 2:]), class_sizes=sizes),
                                       b.add(nat.KIND_ROSS, k, _cols(a[:, :3]), class_sizes=[n])))
    y = np.repeat(np.arange(len(sizes)), sizes)
    w, ref = orc.estimate_semidiscrete_mi(a[:, :2], y, k, detail=True)
    np.testing.assert_array_equal(eps[0], ref["eps"])
    np.testing.assert_array_equal(cnts[0][0], ref["n_full"])
    w, ref = orc.estimate_conditional_semidiscrete_mi(a[:, :1], y, a[:, 2:], k, detail=True)
    np.testing.assert_array_equal(eps[1], ref["eps"])
    for s, key in enumerate(("nxz", "nyz", "nz")):
        np.testing.assert_array_equal(cnts[1][s], ref[key], err_msg=key)


def test_wide_marginals_and_infinities():
    """MI of multi-column variables (counts in both marginals), and infinite
    coordinates in one column."""
    nat = _nat()
    for form in ("plain", "infinite"):
        a = _data(3000, 5, 77, form)
        _both(lambda b: (b.add(nat.KIND_KSG, 3, _cols(a[:, :2]), _cols(a[:, 2:])),
                         b.add(nat.KIND_KSG, 40, _cols(a[:, :1]), _cols(a[:, 4:])),
                         b.add(nat.KIND_KL, 5, _cols(a))))


def test_groups_of_cells():
    """More than 64 cells: boxes of groups."""
    nat = _nat()
    n = 64 * 4096 + 1
    a = _data(n, 4, 5)
    _, eps, cnts = _both(lambda b: b.add(nat.KIND_CMI, 3, _cols(a[:, :1]), _cols(a[:, 1:2]), _cols(a[:, 2:])))
    at = np.random.default_rng(6).integers(0, n, 300)
    pts = np.concatenate([at, [0, n - 1]])
    for i in pts:
        d = np.abs(a - a[i])
        assert eps[0][i] == np.partition(d.max(axis=1), 3)[3]
        r = eps[0][i] - 1e-12
        for s, cols in enumerate(([0, 2, 3], [1, 2, 3], [2, 3])):
            assert cnts[0][s][i] == np.count_nonzero(d[:, cols].max(axis=1) <= r)


@pytest.mark.parametrize("d, n", [(2, 64 * 4096), (2, 64 * 4096 + 1), (3, 16 * 4096), (3, 16 * 4096 + 1), (4, 8 * 4096),
                                  (4, 8 * 4096 + 1), (5, 8 * 4096 + 1)])
def test_cells_by_one_column_or_two(d, n):
    nat = _nat()
    a = _data(n, d, seed=n, form="ties" if n % 2 else "plain")
    if d == 2:
        _both(lambda b: b.add(nat.KIND_KSG, 20, _cols(a[:, :1]), _cols(a[:, 1:])))
    else:
        _both(lambda b: b.add(nat.KIND_CMI, 3, _cols(a[:, :1]), _cols(a[:, 1:2]), _cols(a[:, 2:])))


@pytest.mark.parametrize("k", [3, 4, 7, 8, 15, 16, 31, 32])
@pytest.mark.parametrize("n, m", [(4096, 1), (4097, 1), (8192, 2), (8193, 1), (1000, 40), (1000, 700)])
def test_two_columns_on_trees_or_strips(k, n, m):
    # Both sides of every limit of the two routes, on their own and together.
    nat = _nat()
    a = [_data(n, 2, seed=100 * k + i, form=f) for i, f in enumerate(("plain", "ties", "tails", "equal"))]

    def build(b):
        for i in range(m):
            x = a[i % 4]
            b.add(nat.KIND_KSG, k, _cols(x[:, :1]), _cols(x[:, 1:]))
        b.add(nat.KIND_KL, k, _cols(a[0]))
    _both(build)
