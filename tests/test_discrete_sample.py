"""Columns that a few of their values show not to be countable directly are not
sent to the device for it."""

import numpy as np
import pytest


def _whole(n):
    return np.random.default_rng(n).integers(0, 50, n)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 1000, 16_385])
def test_declined_on_the_host(n, monkeypatch):
    from ennemi_amd import _discrete as d
    monkeypatch.setattr(d.nat, "context", lambda: pytest.fail("sent to the device"))
    a = _whole(n)
    for cols in ([a + 2**53], [a.astype(float) - 2.0**54], [a + 0.5], [a, a + 0.25], [np.full(n, np.nan)], [np.full(n, np.inf)], [a, np.full(n, -np.inf)]):
        assert d._count_rows(cols) is None
    if n > 1:
        far = np.where(np.arange(n) % 2, 70_000, 0)
        assert d._count_rows([far]) is None
        assert d._count_rows([far[::-1].astype(float)]) is None
        assert d._count_rows([np.where(np.arange(n) % 2, 32_768, 0)]) is None
        half = np.where(np.arange(n) % 2, 299, 0)
        assert d._count_rows([half, half]) is None


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 1000, 16_385])
@pytest.mark.parametrize("kind", [np.bool_, np.uint8, np.int8, np.int64, np.float32, np.float64])
def test_countable(n, kind):
    from ennemi_amd import _discrete as d
    a = _whole(n).astype(kind)
    assert d.countable([a], 50) and d.countable([a, a[::-1]], 2500)
    # 256 x 256 is the most.
    wide = np.where(np.arange(n) % 2, 255, 0).astype(np.int64)
    assert d.countable([wide, wide], 256 * 256)


@pytest.mark.parametrize("discrete_x", [False, True])
def test_class_labels(discrete_x, monkeypatch):
    from ennemi_amd import _driver
    monkeypatch.setattr(_driver.nat, "context", lambda: None)
    n = 1000
    a, cont = _whole(n), np.random.default_rng(0).normal(size=n)

    def eligible(labels):
        return _driver._classes_eligible(*((labels, cont) if discrete_x else (cont, labels)), None, discrete_x)

    assert eligible(a) and eligible(a.astype(np.float32)) and eligible(a > 3) and eligible(a + 2**40)
    assert eligible(np.column_stack([a, a])) or not discrete_x
    monkeypatch.setattr(_driver.nat, "context", lambda: pytest.fail("sent to the device"))
    for labels in (a * 0.5 + 0.25, a * 1000, a.astype(str), np.where(a > 3, np.nan, 1.0), a[:0]):
        assert not eligible(labels)
    if discrete_x:
        assert not eligible(np.column_stack([a, a + 0.5]))
