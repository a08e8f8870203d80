"""Class labels prepared and grouped on the device: values, warnings and
errors of the host path, and the grouped columns bit for bit, at the edges of
blocks (2,048 rows) and label ranges."""

import numpy as np
import pytest

from tests.test_gpu_pairs import _caught

pytestmark = pytest.mark.gpu


def _host(monkeypatch, f):
    from ennemi_amd import _driver
    with monkeypatch.context() as m:
        m.setattr(_driver, "_classes_eligible", lambda *a: False)
        return f()


def _both(monkeypatch, on_device, *args, **kw):
    import ennemi_amd as em
    from ennemi_amd import _driver
    used = []
    plan = _driver._plan_classes_device
    with monkeypatch.context() as m:
        m.setattr(_driver, "_plan_classes_device", lambda *a: used.append(plan(*a)) or used[-1])
        got, w = _caught(lambda: em.estimate_mi(*args, **kw))
    ref, wr = _host(monkeypatch, lambda: _caught(lambda: em.estimate_mi(*args, **kw)))
    np.testing.assert_array_equal(got, ref)
    assert w == wr
    assert (bool(used) and used[0] is not None) == on_device


def _labels(rng, n, classes):
    y = rng.integers(0, classes, n)
    y[:1] = 0
    y[-1:] = classes - 1
    return y


@pytest.mark.parametrize("n", [9, 64, 2047, 2048, 2049, 20_000])
@pytest.mark.parametrize("classes", [1, 2, 5, 65])
def test_sizes_and_classes(monkeypatch, n, classes):
    rng = np.random.default_rng(n + classes)
    y = _labels(rng, n, classes)
    x = rng.normal(size=(n, 2)) + y[:, None]
    for kw in ({"discrete_y": True}, {"discrete_y": True, "cond": rng.normal(size=(n, 2))},
               {"discrete_y": True, "preprocess": False, "k": 2}):
        _both(monkeypatch, True, y, x, **kw)
    _both(monkeypatch, True, x[:, 0], np.column_stack((y, y[::-1])), discrete_x=True)


@pytest.mark.parametrize("case", ["lags", "mask", "drop_nan", "cond_lag", "constant", "nan", "short", "bool",
                                  "float_labels", "far_apart", "fractions", "many", "empty_class"])
def test_options_and_errors(monkeypatch, case):
    rng = np.random.default_rng(5)
    n = 3000
    y = _labels(rng, n, 7) - 3
    x = rng.normal(size=(n, 3)) * [1.0, 1e-4, 1e6] + y[:, None]
    kw = {"discrete_y": True}
    lag = 0
    on_device = True
    if case == "lags":
        lag = [-4, 0, 9]
    elif case == "mask":
        kw["mask"] = rng.random(n) < 0.4
    elif case in ("drop_nan", "nan"):
        x[rng.integers(0, n, 300), 1] = np.nan
        kw["drop_nan"] = case == "drop_nan"
        on_device = case == "drop_nan"
    elif case == "cond_lag":
        kw["cond"] = rng.normal(size=(n, 2))
        kw["cond_lag"] = [1, 2]
        lag = [0, 3]
    elif case == "constant":
        x[:, 1] = 4.0
    elif case == "short":
        kw["k"] = n
        on_device = False
    elif case == "bool":
        y = y > 0
    elif case == "float_labels":
        y = y.astype(np.float32)
    elif case == "far_apart":
        y = y * 10_000_000
        on_device = False
    elif case == "fractions":
        y = y / 4
        on_device = False
    elif case == "many":
        y = np.arange(n) % 1000
    elif case == "empty_class":
        y[y == 1] = 2
        kw["mask"] = y != -3
    _both(monkeypatch, on_device, y, x, lag, **kw)


def test_more_classes_than_counters(monkeypatch):
    rng = np.random.default_rng(8)
    for classes, on_device in ((1024, True), (1025, False)):
        y = _labels(rng, 9000, classes)
        _both(monkeypatch, on_device, y, rng.normal(size=9000), discrete_y=True)
