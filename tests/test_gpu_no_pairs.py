"""Tables without a column, or a pair of columns, to estimate."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [0, 1])
@pytest.mark.parametrize("option", [{}, {"mask": True}, {"drop_nan": True}, {"cond": True}])
def test_tables_without_pairs(columns, option):
    from ennemi_amd._driver import plan_pairwise_mi
    n = 30
    rng = np.random.default_rng(1)
    kw = dict(option)
    if "mask" in kw:
        kw["mask"] = np.ones(n, dtype=bool)
    if "cond" in kw:
        kw["cond"] = rng.normal(size=n)
    batch, pairs = plan_pairwise_mi(rng.normal(size=(n, columns)), **kw)
    assert len(batch) == 0 and pairs == []


def test_no_columns_at_all():
    import ennemi_amd
    assert ennemi_amd.pairwise_mi(np.empty((30, 0))).shape == (0, 0)
    y = np.arange(30) % 3
    assert ennemi_amd.estimate_mi(y, np.empty((30, 0)), discrete_y=True).shape == (1, 0)
    assert ennemi_amd.estimate_mi(y + 0.5, np.empty((30, 0), dtype=int), discrete_x=True).shape == (1, 0)
