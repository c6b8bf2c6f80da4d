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
