"""Columns sorted as a whole beside many short classes of theirs: the classes
are sorted in smaller tiles, at the numbers and lengths where that changes."""

import numpy as np
import pytest

from oracle import ennemi_oracle as orc

pytestmark = pytest.mark.gpu


def _nearest(a):
    s = np.sort(a)
    gap = np.concatenate([[np.inf], np.diff(s), [np.inf]])
    d = np.empty(len(a))
    d[np.argsort(a, kind="stable")] = np.minimum(gap[:-1], gap[1:])
    return d


@pytest.mark.parametrize("sizes", [[3] * 255, [3] * 256, [3] * 3000, [1, 2, 511, 512, 513] * 60, [512] * 255 + [513] * 255,
                                   [513] * 256, [600, 2048] * 140, [2049, 8193] * 2 + [5, 700] * 130, [1] * 700 + [8193]])
def test_radii_and_counts_of_classes(sizes):
    import ennemi_amd._native as nat
    from ennemi_amd._batch import Batch
    rng = np.random.default_rng(len(sizes))
    sizes = np.asarray(sizes)
    n = int(sizes.sum())
    label = np.repeat(np.arange(len(sizes)), sizes)
    x = rng.normal(size=n) + 0.1 * (label % 5)
    x[rng.random(n) < 0.3] = 0.5
    b = Batch()
    b.add(nat.KIND_ROSS, 1, [x], class_sizes=sizes)
    value, eps, counts = b.run(export=True)
    first = np.concatenate([[0], np.cumsum(sizes)])
    want = np.concatenate([_nearest(x[a:e]) for a, e in zip(first[:-1], first[1:])])
    np.testing.assert_array_equal(eps[0], want)
    np.testing.assert_array_equal(counts[0][0], orc.ball_counts(x, x, want - 1e-12, backend="kdtree"))
