"""The fused depthwise + pointwise kernel under clamps narrower than a byte, under scales that are powers of two (every channel has exact
ties) and with a depthwise weight zero point at the end of its range, with and without ties; batches with four and with two wavefronts a
tile. Exact against the oracle's two operators."""
import numpy as np
import pytest

import test_gpu_dwpw as DP

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, stride
    (2, 20, 16, 56, 24, 1),
    (2, 36, 8, 40, 40, 2),
    (80, 8, 28, 32, 12, 2),   # a depthwise pass of 8 threads, 560 tiles or more: two wavefronts
    (80, 68, 28, 48, 10, 2),  # ... of more than 128 threads: four
]


def _pow2(s):
    return None if s is None else np.exp2(np.round(np.log2(np.asarray(s, np.float64)))).astype(np.float32)


@pytest.mark.parametrize("what", ["clamp", "ties", "end", "ties_end"])
@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_flavours(oracle, monkeypatch, ci, mode, what):
    if "end" in what and mode != "u8":
        pytest.skip("int8 weights have no zero point")
    pair = DP._pair

    def altered(*args):
        x, wd, bd, kd, wp, bp, kp = pair(*args)
        for k in (kd, kp):
            if what == "clamp":
                k["out_q"] = (k["out_q"][0], 10 if mode == "u8" else -20)
            if "ties" in what:
                k["in_q"] = (float(_pow2(k["in_q"][0])), k["in_q"][1])
                k["w_q"] = (float(_pow2(k["w_q"][0])), k["w_q"][1], _pow2(k["w_q"][2]))
                k["out_q"] = (float(_pow2(k["out_q"][0])), k["out_q"][1])
        if "end" in what:
            kd["w_q"] = (kd["w_q"][0], 0, None)
            kd["in_q"] = (kd["in_q"][0] / 2, kd["in_q"][1])
        kp["in_q"] = kd["out_q"]
        return x, wd, bd, kd, wp, bp, kp
    monkeypatch.setattr(DP, "_pair", altered)
    monkeypatch.setattr(DP, "CASES", CASES)
    DP.test_depthwise_pointwise_fused(oracle, ci, mode, ci % 2)
