"""Columns sent to the device: every type, layout and division into pieces."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.int64, np.int32, np.uint8, np.bool_, ">f8"])
@pytest.mark.parametrize("layout", ["column", "strided", "rows", "columns", "reversed", "one"])
@pytest.mark.parametrize("short", [True, False])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
def test_values_arrive(monkeypatch, dtype, layout, n, short):
    import torch
    from ennemi_amd import _batch, _native as nat
    monkeypatch.setattr(_batch, "_PIECE", 64)
    monkeypatch.setattr(_batch, "_SHORT", 1 << 14 if short else 0)
    rng = np.random.default_rng(n)
    a = (rng.normal(size=(n, 6)) * 1e3).astype(dtype)
    if dtype is np.int64:
        a[0, 0] = 2**62 + 1   # not a double
    a = {"column": a[:, 0].copy(), "strided": a[:, 0], "rows": a, "columns": np.asfortranarray(a),
         "reversed": a[::-1, ::-2], "one": a[:, :1]}[layout]
    ctx = nat.context()
    st = _batch._stream()
    d, pinned = _batch.upload_columns([a, a], torch.device("cuda", ctx.device), st)
    st.synchronize()
    want = np.asarray(a, dtype=np.float64).reshape(n, -1).T.reshape(-1)
    np.testing.assert_array_equal(d.cpu().numpy(), np.concatenate([want, want]))


@pytest.mark.parametrize("nlag, nvar, n, dz, pays", [(97, 8, 3_866, 0, True), (97, 8, 3_865, 0, False), (32, 1, 93_750, 0, True),
                                                     (31, 1, 300_000, 0, False), (97, 8, 100_096, 1, False)])
def test_sort_hints_rule(nlag, nvar, n, dz, pays):
    from ennemi_amd._driver import _hints_pay
    assert _hints_pay(nlag, nvar, n, dz) is pays


def test_estimates_with_and_without_hints(monkeypatch):
    from ennemi_amd import _driver, estimate_mi
    rng = np.random.default_rng(3)
    y, x = rng.normal(size=4_000), rng.normal(size=(4_000, 2))
    x[rng.random(4_000) < 0.1, 1] = np.nan
    got = []
    for pays in (True, False):
        monkeypatch.setattr(_driver, "_hints_pay", lambda *a: pays)
        got.append(estimate_mi(y, x, lag=[-1, 0, 5], drop_nan=True))
    np.testing.assert_array_equal(got[0], got[1])


def test_pinned_memory_is_bounded(monkeypatch):
    import torch
    from ennemi_amd import _batch, _native as nat
    monkeypatch.setattr(_batch, "_PIECE", 4096)
    most = _batch._PIECES * _batch._PIECE
    rng = np.random.default_rng(5)
    table = rng.normal(size=(3 * most // 8 + 5, 8))
    for arrays in ([table[:, 0].copy(), table, rng.integers(0, 9, 2 * most + 1)], [table[::2, ::2], table.T.copy().T]):
        st = _batch._stream()
        d, pinned = _batch.upload_columns(arrays, torch.device("cuda", nat.context().device), st)
        assert pinned.numel() <= most
        st.synchronize()
        want = np.concatenate([np.asarray(a, dtype=np.float64).reshape(len(a), -1).T.reshape(-1) for a in arrays])
        np.testing.assert_array_equal(d.cpu().numpy(), want)


def test_many_columns_share_pieces(monkeypatch):
    import torch
    from ennemi_amd import _batch, _native as nat
    monkeypatch.setattr(_batch, "_PIECE", 1000)
    monkeypatch.setattr(_batch, "_SHORT", 0)
    rng = np.random.default_rng(6)
    cols = [rng.normal(size=n) for n in (1, 999, 1000, 1001, 7, 13, 3000, 1)] + [rng.normal(size=(40, 9))[:, 2]]
    sent = []
    send = torch.Tensor.copy_
    monkeypatch.setattr(torch.Tensor, "copy_", lambda self, *a, **k: (sent.append(len(self)), send(self, *a, **k))[1])
    d, _ = _batch.upload_columns(cols, torch.device("cuda", nat.context().device), _batch._stream())
    monkeypatch.undo()
    torch.cuda.synchronize()
    want = np.concatenate(cols)
    np.testing.assert_array_equal(d.cpu().numpy(), want)
    assert sent == [1000] * (len(want) // 1000) + [len(want) % 1000]
