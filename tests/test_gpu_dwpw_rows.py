"""The fused depthwise + pointwise kernel with one, two and four output rows a tile, whichever its own rule would take, where its
pieces end: rows that leave a partial sixteen-pixel store (28 and 20 wide), an odd number of pixel tiles taken two at a time (at most
16 channels in the last tile), pointwise weights too large to be copied to LDS, a depthwise weight zero point at the end of
its range, the first and the last bytes of the input tensor. Exact against the oracle's two operators."""
import pytest

import test_gpu_dwpw as DP

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, stride
    (1, 8, 4, 28, 16, 1),
    (2, 36, 4, 20, 48, 1),
    (1, 33, 8, 56, 1, 2),
    (2, 24, 16, 40, 10, 2),
    (3, 4, 4, 4, 17, 1),
    (1, 256, 4, 16, 320, 1),
    (1, 256, 8, 32, 320, 2),
]


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8zp0"])
@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_rows(oracle, monkeypatch, ci, rows, mode):
    monkeypatch.setenv("TVX_DWPW_ROWS", str(rows))
    monkeypatch.setattr(DP, "CASES", CASES)
    if mode == "u8zp0":
        pair = DP._pair

        def shifted(*args):
            x, wd, bd, kd, wp, bp, kp = pair(*args)
            kd["w_q"] = (kd["w_q"][0], 0, None)
            # (every tap counts 120-odd more: a finer input scale keeps the results as spread as before)
            kd["in_q"] = (kd["in_q"][0] / 2, kd["in_q"][1])
            return x, wd, bd, kd, wp, bp, kp
        monkeypatch.setattr(DP, "_pair", shifted)
    DP.test_depthwise_pointwise_fused(oracle, ci, "u8" if mode == "u8zp0" else mode, 1 if ci % 2 else 0)


@pytest.mark.parametrize("n,c,h,w,oc", [(8, 288, 128, 128, 64), (8, 224, 112, 112, 256), (8, 256, 128, 128, 96), (16, 352, 80, 80, 128)])
def test_as_many_rows_as_fit(oracle, n, c, h, w, oc):
    """Pairs whose four rows a tile do not fit LDS, though fewer do: taken with those."""
    import numpy as np
    import torch
    import tvx_case as TC
    rng = np.random.default_rng(8100 + c)
    x, wd, bd, kd, wp, bp, kp = DP._pair(rng, n, c, h, w, oc, 1, "i8pc")
    T, keep = TC.tvx(), []
    op = T.conv2d_dw_pw_create(DP._desc(T, kd, 0, keep), wd, bd, DP._desc(T, kp, 2, keep), wp, bp)
    assert op.kernel_name == "dwconv3x3_pwconv_i8"
    xd, yd = TC.to_device(x), TC.device_out(n * oc * h * w, np.int8)
    op.run(xd, None, yd)
    torch.cuda.synchronize()
    got = yd.cpu().numpy().reshape(n, -1)
    op.close()
    for image in (0, n - 1):   # (the oracle takes seconds for one)
        for k in (kd, kp):
            k["in_shape"][3] = k["out_shape"][3] = 1
        mid = oracle.conv2d(x.reshape(n, -1)[image].copy(), wd, bd, act=0, **kd)
        want = oracle.conv2d(mid, wp, bp, act=2, **kp)
        assert np.array_equal(got[image], want), (image, int((got[image] != want).sum()))
