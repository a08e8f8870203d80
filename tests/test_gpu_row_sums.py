"""Mean and deviation of the columns of a condition of several columns: the
device adds them in tiles, the host plan row by row (NumPy's axis=0 order).
The rescaled columns must be the same bits.

The data take every way through a tile: sums that stay in one binade, that
cross many, that change sign; additions that are ties for most rows, with the
sum even or odd; rows of zeros; cancellation."""

import numpy as np
import pytest

from tests.test_gpu_prep import _compare

pytestmark = pytest.mark.gpu


def _column(kind, n, rng):
    z = rng.normal(size=n)
    if kind == "offset":
        return z + 1e6
    if kind == "walk":
        return np.sign(z)
    if kind == "low bits":
        return 1.0 + rng.integers(0, 4, n) * 2.0**-52
    if kind in ("ties", "negative ties"):   # the sum's unit is 2**-22
        v = rng.integers(-3, 4, n) * 2.0**-23
        v[0] = 2.0**30 * (1 if kind == "ties" else -1) * 1.25
        return v
    if kind == "edge":   # about the lower end of a binade
        v = rng.integers(-3, 4, n) * 2.0**-23
        v[0] = 2.0**30
        return v
    if kind == "growing":
        return z * np.exp(np.linspace(-30.0, 30.0, n))
    if kind == "cancelling":
        return np.where(np.arange(n) % 2 == 0, 1e16, -1e16) + z
    if kind == "zeros":
        v = np.zeros(n)
        v[n // 2:] = z[n // 2:]
        return v
    if kind == "constant":
        return np.full(n, 0.1)
    return z


KINDS = ["normal", "offset", "walk", "low bits", "ties", "negative ties", "edge", "growing", "cancelling", "zeros",
         "constant"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1000, 16_383, 16_384, 16_385, 16_384 + 64, 20_480 - 1, 20_480 + 65, 100_003])
def test_row_sums(kind, n):
    rng = np.random.default_rng([n, KINDS.index(kind)])
    cond = np.column_stack([_column(kind, n, rng), rng.normal(size=n), -_column(kind, n, rng)])
    y, x = rng.normal(size=(2, n))
    _compare((y, x, 0), dict(k=3, cond=cond))


def test_many_columns_of_several_tasks():
    rng = np.random.default_rng(2)
    n = 40_000
    y, cond = rng.normal(size=n), rng.normal(size=(n, 2)) + [0.0, 3.0]
    x = rng.normal(size=(n, 2))
    x[rng.random(n) < 0.3, 1] = np.nan
    _compare((y, x, [0, 1, -700]), dict(k=3, cond=cond, drop_nan=True, mask=rng.random(n) < 0.9))
