"""The convolution + 2 x 2 MAX pooling kernel for planes that fit LDS, with its reduction whole and split, its tiles in one workgroup and in several: channel counts around a
step, padding on every side, strides and dilation, rows of four to nine columns, more pixel tiles than wavefronts, pooled planes that
end inside a tile, a weight zero point at the end of its range. Exact against the oracle's two operators."""
import pytest

import test_gpu_fused_small_nets as SN
import tvx_case as TC

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=2, c=17, h=12, w=12, oc=33, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[0, 0, 0, 0]),
    dict(n=1, c=64, h=9, w=4, oc=20, kh=2, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 0, 0]),
    dict(n=3, c=33, h=8, w=9, oc=24, kh=3, kw=4, stride=[1, 2], dil=[1, 1], pad=[1, 1, 1, 0]),
    dict(n=1, c=32, h=24, w=20, oc=40, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1]),    # fifteen tiles
    dict(n=2, c=16, h=8, w=9, oc=32, kh=3, kw=2, stride=[1, 1], dil=[3, 2], pad=[0, 0, 1, 1]),
    dict(n=1, c=100, h=3, w=6, oc=70, kh=2, kw=1, stride=[1, 1], dil=[1, 1], pad=[0, 0, 0, 0]),     # one step a part
]


@pytest.mark.parametrize("mode", ["u8", "u8zp0"])
@pytest.mark.parametrize("groups", [1, 2, 7, 99])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_tiles_dealt_out_to_workgroups(oracle, monkeypatch, ci, groups, mode):
    """Each loads the rows behind its own tiles."""
    monkeypatch.setenv("TVX_CONV_POOL_GROUPS", str(groups))
    _run(oracle, monkeypatch, ci, mode)


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8zp0"])
@pytest.mark.parametrize("parts", [1, 3, 8])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_split_reductions(oracle, monkeypatch, ci, parts, mode):
    monkeypatch.setenv("TVX_CONV_POOL_PARTS", str(parts))
    _run(oracle, monkeypatch, ci, mode)


def _run(oracle, monkeypatch, ci, mode):
    monkeypatch.setattr(SN, "CONV_POOL", [dict(c, kernel="conv2d_igemm_maxpool_i8") for c in CASES])
    case = SN.conv_case

    def fitted(*args, **kws):
        x, w, b, kws = case(*args, **kws)
        if mode == "u8zp0":   # (every weight counts 120-odd more)
            kws["w_q"] = (kws["w_q"][0], 0, None)
            kws["out_q"] = (kws["out_q"][0] * 2, kws["out_q"][1])
        kws["in_q"] = (kws["in_q"][0] / 8, kws["in_q"][1])   # (the largest of four results would mostly lie on the clamp)
        return x, w, b, kws
    monkeypatch.setattr(SN, "conv_case", fitted)
    TC.expect_variant(monkeypatch, "conv2d_pool_i8")
    SN.test_conv2d_with_fused_max_pool(oracle, ci, "u8" if mode == "u8zp0" else mode, 0, monkeypatch)
