"""FullyConnected on small tiles (any K; int8, float16, float32): rows, features and reductions that end inside tiles and steps."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import rand_q

pytestmark = pytest.mark.gpu

SIZES = [(1, 16, 1), (1, 800, 10), (3, 33, 17), (16, 64, 16), (17, 65, 31), (33, 1001, 70), (64, 127, 65), (130, 48, 129), (70, 5, 40)]


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8pc", "f16", "f32"])
@pytest.mark.parametrize("m,k,n", SIZES)
def test_fully_connected_rows(oracle, m, k, n, mode, monkeypatch):
    rng = np.random.default_rng(m * 31 + k + n)
    monkeypatch.setenv("TVX_FC_ROWS", "1")
    if mode in ("f16", "f32"):
        npd, dt = (np.float16, 2) if mode == "f16" else (np.float32, 3)
        x, w = rng.standard_normal(m * k).astype(npd), (rng.standard_normal(n * k) / np.sqrt(k)).astype(npd)
        b = rng.standard_normal(n).astype(np.float32)
        kws = dict(m=m, k=k, n=n, in_dtype=dt, w_dtype=dt, out_dtype=dt)
    else:
        in_dt, w_dt = (0 if mode.startswith("u8") else 1), (0 if mode == "u8" else 1)
        x, w = rand_q(rng, m * k, in_dt), rand_q(rng, n * k, w_dt)
        b = rng.integers(-3000, 3001, n).astype(np.int32)
        wq = (0.01, 117, None) if mode == "u8" else (1.0, 0, np.exp(rng.uniform(np.log(0.003), np.log(0.02), n)).astype(np.float32))
        kws = dict(m=m, k=k, n=n, in_dtype=in_dt, w_dtype=w_dt, out_dtype=in_dt, in_q=(0.02, 131 if in_dt == 0 else -2), w_q=wq,
                   out_q=(float(np.float32(0.02 * 0.01 * 40 * np.sqrt(k))), 5 if in_dt == 0 else 0))
    want = oracle.fully_connected(x, w, b, act=1, **kws)
    for shape in range(3):   # 16 x 16, 32 x 32, 64 x 64
        monkeypatch.setenv("TVX_FC_ROWS_SHAPE", str(shape))
        got = TC.gpu_fully_connected(x, w, b, act=1, want_kernel="fc_rows_" + {"f16": "f16", "f32": "f32"}.get(mode, "i8"), **kws)
        if mode in ("f16", "f32"):
            assert np.allclose(got.astype(np.float64), want.astype(np.float64), rtol=2e-3 if mode == "f16" else 1e-5, atol=2e-3 if mode == "f16" else 1e-5), shape
        else:
            assert np.array_equal(got, want), (shape, int((got != want).sum()))


def test_fully_connected_rows_keep_an_infinity_apart(monkeypatch):
    """A row that ends inside a reduction step is not multiplied with the row behind it."""
    monkeypatch.setenv("TVX_FC_ROWS", "1")
    x, w = np.ones((4, 37), np.float32), np.ones((20, 37), np.float32)
    x[2, 0] = np.inf
    got = TC.gpu_fully_connected(x.ravel(), w.ravel(), None, m=4, k=37, n=20, in_dtype=3, w_dtype=3, out_dtype=3, want_kernel="fc_rows_f32").reshape(4, 20)
    assert np.isinf(got[2]).all() and np.array_equal(got[[0, 1, 3]], np.full((3, 20), 37, np.float32))


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("mode", ["u8", "f16"])
def test_fully_connected_rows_of_a_view(oracle, mode, offset, monkeypatch):
    """Rows of whole dwords in a tensor that does not begin on one: the input is a view some elements into a buffer."""
    import torch
    to_device = TC.to_device
    monkeypatch.setattr(TC, "to_device", lambda a: torch.cat([to_device(np.zeros(offset, a.dtype)), to_device(a)])[offset:])
    test_fully_connected_rows(oracle, 33, 96, 70, mode, monkeypatch)
