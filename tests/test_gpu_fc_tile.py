"""FullyConnected on tiles whose rows and weights go through LDS (any K; int8, float16): rows, features and reductions that end
inside tiles, stages and sixteen-byte chunks, rows that begin at any element, one stage and several."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import rand_q

pytestmark = pytest.mark.gpu

SIZES = [(1, 16, 1), (3, 33, 17), (64, 128, 64), (65, 129, 65), (130, 300, 129), (129, 37, 200), (70, 1001, 40), (257, 64, 80), (300, 257, 300)]


def _case(m, k, n, mode):
    rng = np.random.default_rng(m * 37 + k + n)
    if mode == "f16":
        x, w = rng.standard_normal(m * k).astype(np.float16), (rng.standard_normal(n * k) / np.sqrt(k)).astype(np.float16)
        return x, w, rng.standard_normal(n).astype(np.float32), dict(m=m, k=k, n=n, in_dtype=2, w_dtype=2, out_dtype=2)
    in_dt, w_dt = (0 if mode.startswith("u8") else 1), (0 if mode == "u8" else 1)
    x, w = rand_q(rng, m * k, in_dt), rand_q(rng, n * k, w_dt)
    wq = (0.01, 117, None) if mode == "u8" else (1.0, 0, np.exp(rng.uniform(np.log(0.003), np.log(0.02), n)).astype(np.float32))
    return x, w, rng.integers(-3000, 3001, n).astype(np.int32), dict(
        m=m, k=k, n=n, in_dtype=in_dt, w_dtype=w_dt, out_dtype=in_dt, in_q=(0.02, 131 if in_dt == 0 else -2), w_q=wq,
        out_q=(float(np.float32(0.02 * 0.01 * 40 * np.sqrt(k))), 5 if in_dt == 0 else 0))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8pc", "f16"])
@pytest.mark.parametrize("m,k,n", SIZES)
def test_tiles_through_lds(oracle, m, k, n, mode, offset, monkeypatch):
    import torch
    x, w, b, kws = _case(m, k, n, mode)
    monkeypatch.setenv("TVX_FC_ROWS", "1")
    if offset:   # a view some elements into a buffer
        to_device = TC.to_device
        monkeypatch.setattr(TC, "to_device", lambda a: torch.cat([to_device(np.zeros(offset, a.dtype)), to_device(a)])[offset:])
    want = oracle.fully_connected(x, w, b, act=1, **kws)
    TC.expect_variant(monkeypatch, "fc_tile_f16" if mode == "f16" else "fc_tile_i8")
    for shape in range(3, 8):
        monkeypatch.setenv("TVX_FC_ROWS_SHAPE", str(shape))
        got = TC.gpu_fully_connected(x, w, b, act=1, want_kernel="fc_rows_f16" if mode == "f16" else "fc_rows_i8", **kws)
        if mode == "f16":   # (results of a few units, off by up to one unit of float16's last place: 2^-9 at 1 to 2)
            assert np.allclose(got.astype(np.float64), want.astype(np.float64), rtol=2e-3, atol=2e-3), shape
        else:
            assert np.array_equal(got, want), (shape, int((got != want).sum()))


@pytest.mark.parametrize("mode", ["u8", "i8pc", "f16"])
@pytest.mark.parametrize("m,n", [(1, 1), (65, 70), (130, 129), (300, 257)])
@pytest.mark.parametrize("k", [64, 128, 129, 300, 512, 577, 1153])
def test_stages_on_groups(oracle, m, n, k, mode, monkeypatch):
    """Reductions cut over groups of wavefronts: fewer stages than groups, as many, one more, a last round that is not full."""
    x, w, b, kws = _case(m, k, n, mode)
    monkeypatch.setenv("TVX_FC_ROWS", "1")
    want = oracle.fully_connected(x, w, b, act=1, **kws)
    TC.expect_variant(monkeypatch, "fc_tile_f16" if mode == "f16" else "fc_tile_i8")
    monkeypatch.setenv("TVX_FC_ROWS_SHAPE", "8")
    got = TC.gpu_fully_connected(x, w, b, act=1, want_kernel="fc_rows_f16" if mode == "f16" else "fc_rows_i8", **kws)
    if mode == "f16":   # (results of a few units, off by up to one unit of float16's last place: 2^-9 at 1 to 2)
        assert np.allclose(got.astype(np.float64), want.astype(np.float64), rtol=2e-3, atol=2e-3)
    else:
        assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("shape", [3, 5, 7, 8])
def test_rows_keep_an_infinity_apart(monkeypatch, shape):
    """What lies behind a row that ends inside a stage is not multiplied."""
    monkeypatch.setenv("TVX_FC_ROWS", "1")
    monkeypatch.setenv("TVX_FC_ROWS_SHAPE", str(shape))
    TC.expect_variant(monkeypatch, "fc_tile_f16")
    x, w = np.ones((4, 37), np.float16), np.ones((20, 37), np.float16)
    x[2, 0] = np.inf
    got = TC.gpu_fully_connected(x.ravel(), w.ravel(), None, m=4, k=37, n=20, in_dtype=2, w_dtype=2, out_dtype=2, want_kernel="fc_rows_f16").reshape(4, 20)
    assert np.isinf(got[2]).all() and np.array_equal(got[[0, 1, 3]], np.full((3, 20), 37, np.float16))


@pytest.mark.parametrize("m,k,n,mode,kernel", [
    (332, 672, 1965, "i8pc", "fc_rows_i8"), (578, 685, 832, "i8pc", "fc_rows_i8"), (617, 358, 921, "f16", "fc_rows_f16"),   # reductions that end early in their last stage
    (393, 704, 1908, "u8", "fc_tile_i8"), (900, 512, 1100, "f16", "fc_tile_f16"), (3521, 560, 1238, "i8pc", "fc_tile_i8"),
    # up to two 32 x 32 tiles a compute unit (of 256): rows that fit an L2 and are no whole cache lines apart, whole ones, more than fit, rows at odd bytes
    (263, 1168, 1639, "f16", "fc_rows_f16"), (361, 2576, 1124, "i8pc", "fc_rows_i8"), (192, 2752, 2517, "f16", "fc_tile_f16"), (2195, 1888, 163, "f16", "fc_tile_f16"),
    (383, 1098, 1136, "u8", "fc_tile_i8"), (3532, 1696, 127, "i8pc", "fc_rows_i8"), (3468, 1952, 108, "f16", "fc_tile_f16")])
def test_which_tiles_a_layer_gets(oracle, m, k, n, mode, kernel, monkeypatch):
    x, w, b, kws = _case(m, k, n, mode)
    TC.expect_variant(monkeypatch, kernel)
    got, want = TC.gpu_fully_connected(x, w, b, act=1, **kws), oracle.fully_connected(x, w, b, act=1, **kws)
    if mode == "f16":   # (as above)
        assert np.allclose(got.astype(np.float64), want.astype(np.float64), rtol=2e-3, atol=2e-3)
    else:
        assert np.array_equal(got, want)
