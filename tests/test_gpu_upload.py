"""Columns sent to the device: every type, layout and division into pieces."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.int64, np.int32, np.uint8, np.bool_, ">f8"])
@pytest.mark.parametrize("layout", ["column", "strided", "rows", "columns", "reversed", "one"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
def test_values_arrive(monkeypatch, dtype, layout, n):
    import torch
    from ennemi_amd import _batch, _native as nat
    monkeypatch.setattr(_batch, "_PIECE", 64)
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
