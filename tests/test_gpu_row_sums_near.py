"""Row-by-row sums that come close to the ends of a binade at the edges of tiles,
so that tiles are expected to leave it and do not: a condition's columns are
rescaled with NumPy's mean and deviation, bit for bit."""

import numpy as np
import pytest

from tests.test_gpu_prep import _compare

pytestmark = pytest.mark.gpu


def _column(kind, n, rng):
    z = rng.normal(size=n)
    if kind == "near one":            # 2**k after 2**k rows, or a little more or less
        return 1.0 + 1e-13 * z
    if kind == "near minus a half":
        return -0.5 - 3e-14 * z
    if kind == "above":               # always a few units above
        return 1.0 + rng.integers(0, 3, n) * 2.0**-52
    if kind == "steps":               # tiles of very different rows
        return np.repeat(rng.normal(size=n // 64 + 1), 64)[:n] * 1e-3 + 1.0 + 1e-13 * z
    if kind == "whole":
        return 4.0 + rng.integers(-1, 2, n)
    if kind == "lingering":           # about 2**20, up and down, in units of 2**-32
        v = rng.choice([-1.0, 1.0], n) * (2.0**-12 + rng.integers(0, 8, n) * 2.0**-33)
        v[::64] += rng.normal(size=len(v[::64])) * 2.0**-6
        v[0] = 2.0**20
        return v
    return z


KINDS = ["near one", "near minus a half", "above", "steps", "whole", "lingering"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [16_384, 16_385, 19_115, 20_480, 32_768 + 4096, 65_536 + 64, 100_003, 262_144 + 5])
@pytest.mark.parametrize("seed", [0, 1])
def test_row_sums(kind, n, seed):
    rng = np.random.default_rng([n, KINDS.index(kind), seed])
    cond = np.column_stack([_column(kind, n, rng), _column(kind, n, rng) * 2.0**rng.integers(-40, 40), rng.normal(size=n)])
    y, x = rng.normal(size=(2, n))
    _compare((y, x, 0), dict(k=3, cond=cond))
