"""1x1 convolution with a wavefront's pixels in registers: images and batches that end inside pixel groups, channels inside steps and
output tiles, reductions shared by four wavefronts, the Add behind it."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import rand_q

pytestmark = pytest.mark.gpu

# n, c, h, w, oc
SIZES = [(1, 1, 1, 4, 1), (1, 5, 2, 4, 3), (3, 64, 3, 3, 16), (2, 65, 7, 7, 33), (5, 130, 5, 13, 17), (1, 192, 16, 16, 48), (2, 256, 9, 11, 70),
         (3, 300, 7, 7, 20), (1, 512, 4, 4, 100), (2, 577, 3, 5, 40), (40, 24, 13, 13, 144), (1, 2048, 2, 3, 18),
         # channels at the edges of steps of 32 and of 64 and of a lane's 8 and 16; the last images' rows end with the tensor
         (2, 8, 5, 11, 20), (3, 16, 4, 9, 33), (2, 31, 9, 9, 17), (5, 32, 3, 5, 16), (2, 33, 7, 5, 40), (3, 48, 6, 6, 16), (2, 129, 5, 5, 20)]


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8pc", "i8big"])
@pytest.mark.parametrize("n,c,h,w,oc", SIZES)
def test_pointwise_in_registers(oracle, n, c, h, w, oc, mode, monkeypatch):
    rng = np.random.default_rng(n * 7 + c + h * w + oc)
    in_dt, w_dt = (0 if mode.startswith("u8") else 1), (0 if mode == "u8" else 1)
    x, wt = rand_q(rng, n * c * h * w, in_dt), rand_q(rng, oc * c, w_dt)
    b = rng.integers(-3000, 3001, oc).astype(np.int32)
    wq = (0.0123, 117, None) if mode == "u8" else (1.0, 0, np.exp(rng.uniform(np.log(0.003), np.log(0.02), oc)).astype(np.float32))
    in_q, out_q = (0.0211, 131 if in_dt == 0 else -2), (float(np.float32(0.0217 * 0.0123 * 40 * np.sqrt(c))), 5 if in_dt == 0 else 0)
    if mode == "i8big":   # multipliers of .25 to 2, small codes: powers of two among them, so that ties occur
        x, wt, b = (x // 32).astype(np.int8), (wt // 32).astype(np.int8), b // 100
        wq = (1.0, 0, np.array([0.25, 0.5, 0.31, 1.0, 1.7, 0.75])[np.arange(oc) % 6].astype(np.float32))
        in_q, out_q = (1.0, -2), (1.0, 3)
    kws = dict(in_shape=[w, h, c, n], w_shape=[1, 1, c, oc], out_shape=[w, h, oc, n], stride=[1, 1], dilation=[1, 1], pad_left=0, pad_top=0,
               multiplier=0, in_dtype=in_dt, w_dtype=w_dt, out_dtype=in_dt, in_q=in_q, w_q=wq, out_q=out_q)
    want = [oracle.conv2d(x, wt, b, act=act, **kws) for act in (0, 1)]
    ran = 0
    for form, most, px in (("1", 256, 8), ("4", 2048, 4)):
        for waves in ("1", "100000"):   # every output tile in one wavefront; each in its own
            if c > most or h * w < px:
                continue
            monkeypatch.setenv("TVX_PWCONV_REG", form)
            monkeypatch.setenv("TVX_PWCONV_REG_WAVES", waves)
            for act in (0, 1):
                got = TC.gpu_conv2d(x, wt, b, act=act, want_kernel="pwconv_reg_i8", **kws)
                assert np.array_equal(got, want[act]), (form, waves, act, int((got != want[act]).sum()))
            ran += 1
    assert ran


@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("n,side", [(64, 7), (9, 13), (3, 10)])
def test_add_written_over_its_operand(oracle, n, side, mode, monkeypatch):
    """The fused Add with its result in the buffer of its other operand: planes whose last pixel group overlaps the one before."""
    import test_gpu_parity as P
    made, to_device = [], TC.to_device
    monkeypatch.setattr(TC, "to_device", lambda a: made.append(to_device(a)) or made[-1])
    monkeypatch.setattr(TC, "device_out", lambda count, dtype: made[-1])   # the operand, uploaded last
    P.test_pointwise_conv_with_fused_add(oracle, side, n, mode, 2)
