"""Calls with little to prepare, which are prepared on the host: the limits, and
the same values on both sides of them."""

import numpy as np
import pytest

from tests.test_gpu_classes import _both, _labels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kept,on_device", [(4096, None, False), (4097, None, True), (9000, 4096, False),
                                              (9000, 4097, True), (40, None, False)])
@pytest.mark.parametrize("option", [{}, {"preprocess": False}, {"cond": True}])
def test_one_estimate_against_classes(monkeypatch, n, kept, on_device, option):
    rng = np.random.default_rng(n)
    y = _labels(rng, n, 4)
    kw = dict(option)
    if "cond" in kw:
        kw["cond"] = rng.normal(size=n)
    if kept is not None:
        kw["mask"] = np.isin(np.arange(n), rng.permutation(n)[:kept])
    _both(monkeypatch, on_device, y, rng.normal(size=n) + y, discrete_y=True, **kw)
    _both(monkeypatch, on_device, rng.normal(size=n) + y, y, discrete_x=True, **kw)


@pytest.mark.parametrize("n,m,option,on_device", [
    (3000, 2, {}, False), (3001, 2, {}, True), (40, 3, {}, True), (3000, 2, {"mask": 3000}, False),
    (9000, 2, {"mask": 3001}, True), (500, 5, {"preprocess": False}, False), (500, 6, {"preprocess": False}, True),
    (30_001, 2, {"preprocess": False}, True), (30_000, 2, {"preprocess": False}, False)])
def test_pairs(monkeypatch, n, m, option, on_device):
    import ennemi_amd as em
    from ennemi_amd import _driver
    rng = np.random.default_rng(n)
    data = rng.normal(size=(n, m))
    kw = dict(option)
    if "mask" in kw:
        kw["mask"] = np.isin(np.arange(n), rng.permutation(n)[:kw["mask"]])
    used = []
    plan = _driver._plan_pairwise_device
    with monkeypatch.context() as c:
        c.setattr(_driver, "_plan_pairwise_device", lambda *a: used.append(1) or plan(*a))
        got = em.pairwise_mi(data, **kw)
    assert bool(used) == on_device
    with monkeypatch.context() as c:
        c.setattr(_driver, "_pairs_sooner_on_host", lambda *a: on_device)   # the other way
        np.testing.assert_array_equal(em.pairwise_mi(data, **kw), got)


@pytest.mark.parametrize("spoil", ["constant", "two", "nearly", "masked"])
def test_constant_columns(monkeypatch, spoil):
    import warnings

    import ennemi_amd as em
    from ennemi_amd import _driver
    rng = np.random.default_rng(3)
    data = rng.normal(size=(700, 4))
    data[:, 2] = 1.5
    kw = {}
    if spoil == "two":
        data[:, 0] = 0.0
    elif spoil == "nearly":
        data[123, 2] = 1.75
    elif spoil == "masked":
        kw["mask"] = rng.random(700) < 0.5
    used = []
    plan = _driver._plan_pairwise_device
    with monkeypatch.context() as c, warnings.catch_warnings():
        warnings.simplefilter("ignore")
        c.setattr(_driver, "_plan_pairwise_device", lambda *a: used.append(1) or plan(*a))
        got = em.pairwise_mi(data, **kw)
        assert bool(used) == (spoil in ("nearly", "masked"))
        c.setattr(_driver, "_device_prep_arrays", lambda *a: False)
        np.testing.assert_array_equal(em.pairwise_mi(data, **kw), got)
