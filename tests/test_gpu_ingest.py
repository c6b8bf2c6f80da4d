"""Transpose and DataConvert: each way a permutation is moved, at its edges, with pointers of any alignment; counts that end inside
four elements, ties and values with no number."""
import numpy as np
import pytest

import tvx_case as TC

pytestmark = pytest.mark.gpu

# interleaved (few channels, runs past a chunk), tiles (edges of 64), gathers (rows of any width), several batch dimensions, 4 others
MOVES = [((3, 2731, 2), (1, 0, 2), "interleaved"), ((1, 3, 5), (1, 2, 0), "gather"), ((16, 513), (1, 0), "interleaved"), ((3, 7, 5, 4, 3), (1, 0, 4, 2, 3), "interleaved"),
         ((65, 64), (1, 0), "tiles"), ((130, 67, 3), (1, 0, 2), "tiles"), ((2, 63, 129), (2, 1, 0), "tiles"), ((66, 3, 65, 2, 2), (2, 4, 3, 1, 0), "tiles"),
         ((6, 5, 4), (0, 2, 1), "gather"), ((16, 9, 7), (0, 2, 1), "gather"), ((2, 3, 2, 3, 2, 3), (1, 0, 3, 2, 5, 4), "gather")]


@pytest.mark.parametrize("dt", [np.uint8, np.float16, np.int32])
@pytest.mark.parametrize("in_dims,perm,form", MOVES)
def test_transpose_forms(oracle, in_dims, perm, form, dt, variant=None):
    import torch
    T, n = TC.tvx(), int(np.prod(in_dims))
    if dt == np.int32 and in_dims[0] in (16,) and form == "interleaved":
        assert in_dims[0] * 4 == 64   # the widest pixel of that form
    x = (np.arange(n) * 7 + 3).astype(np.uint32).astype(np.uint8 if dt == np.uint8 else np.int16 if dt == np.float16 else dt).view(dt)
    want = oracle.transpose(x, in_dims, perm)
    d = T.TransposeDesc()
    d.rank, d.elem_bytes = len(in_dims), x.dtype.itemsize
    for i, (e, p) in enumerate(zip(in_dims, perm)):
        d.in_dims[i], d.perm[i] = e, p
    op = T.transpose_create(d)
    assert op.kernel_name == "transpose_" + form
    assert variant is None or op.variant == op.kernel_name + variant, op.variant
    e = x.dtype.itemsize
    for off in (0, 1, 2):   # elements
        xd, yd = torch.zeros((n + 8) * e, dtype=torch.uint8, device="cuda"), torch.full(((n + 8) * e,), 0xA5, dtype=torch.uint8, device="cuda")
        xd[off * e:(off + n) * e] = torch.from_numpy(x.view(np.uint8).copy()).cuda()
        op.run(xd.data_ptr() + off * e, None, yd.data_ptr() + off * e)
        torch.cuda.synchronize()
        y = yd.cpu().numpy()
        assert np.array_equal(y[off * e:(off + n) * e], want.view(np.uint8)), off
        assert (y[:off * e] == 0xA5).all() and (y[(off + n) * e:] == 0xA5).all(), off


# up to eight channels sorted in registers: around a thread's pixels (8 bytes, 4 halves, 2 words), a workgroup's, and with two batch dimensions; more
# through LDS in blocks or one by one: around a workgroup's pixels and a block's
FEW = [((a, b, 3), (1, 0, 2), "interleaved") for a in range(2, 9) for b in (2, 7, 8, 9, 511, 2051)] + \
      [((a, 11, 3, 2), (1, 0, 3, 2), "interleaved") for a in (2, 3, 8, 12)] + [((3, 2048, 2), (1, 0, 2), "interleaved")] + \
      [((a, b, 2), (1, 0, 2), "interleaved") for a in (9, 10, 12, 16) for b in (2, 3, 255, 509, 681, 683)]


@pytest.mark.parametrize("dt", [np.uint8, np.float16, np.int32])
@pytest.mark.parametrize("in_dims,perm,form", FEW)
def test_transpose_of_few_channels(oracle, in_dims, perm, form, dt):
    e, (channels, pixels) = np.dtype(dt).itemsize, in_dims[:2]
    blocks = channels % 4 == 0 and e <= 2 and pixels >= 4 // e
    test_transpose_forms(oracle, in_dims, perm, form, dt, "_reg" if channels <= 8 and pixels >= 8 // e else "_block" if blocks else "")


@pytest.mark.parametrize("channels,dt", [(20, np.uint8), (32, np.uint8), (60, np.uint8), (64, np.uint8), (20, np.float16), (32, np.float16), (18, np.float16)])
@pytest.mark.parametrize("pixels", [3, 4, 5, 126, 128, 129, 130, 131, 410])
def test_transpose_of_wide_pixels(oracle, pixels, channels, dt):
    test_transpose_forms(oracle, (channels, pixels, 3), (1, 0, 2), "interleaved", dt, "" if channels == 18 or (pixels == 3 and dt == np.uint8) else "_block")


@pytest.mark.parametrize("out_dt", [0, 1, 2, 3])
@pytest.mark.parametrize("in_dt", [0, 1, 2, 3])
@pytest.mark.parametrize("count", [1, 3, 4, 1021, 4099])
def test_convert_edges(oracle, count, in_dt, out_dt):
    rng = np.random.default_rng(count * 16 + in_dt * 4 + out_dt)
    for scale in (0.1, 0.0078125, 1e-39):   # no tie is exact; every other input is one; a reciprocal that is no float
        if in_dt < 2:
            x = rng.integers(-128, 128, count).astype(np.int8).view(TC.NP_OF[in_dt])
        else:
            x = (rng.integers(-600, 600, count) * 0.5 * scale).astype(np.float32)
            x[::5] = np.nextafter(x[::5], np.float32(np.inf))
            if count > 100 and out_dt >= 2:
                x[7], x[11] = np.inf, -np.inf
            x = x.astype(TC.NP_OF[in_dt])
        q_in = (float(np.float32(scale)) if in_dt < 2 else 1.0, 3 if in_dt < 2 else 0)
        args = (in_dt, q_in, out_dt, (float(np.float32(scale)), 128 if out_dt == 0 else -5))
        with np.errstate(all="ignore"):
            want = oracle.convert(x, *args)
        assert np.array_equal(TC.gpu_convert(x, *args), want, equal_nan=True), scale
