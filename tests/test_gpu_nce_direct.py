"""The form of the convolutions and matmuls that stages nothing (nce_direct): every tile and wave count at its edges, and
the families' own kernels on the small layers it otherwise serves."""
import numpy as np
import pytest

from test_gpu_nce_views import FAMILIES, run_views, seed

pytestmark = pytest.mark.gpu

LAYERS = [
    # one row; channels that are no multiple of 4, 16; K of one 16-byte chunk, of a remainder, of more steps than waves
    dict(N=1, H=1, W=1, IC=16, OC=1, KY=1, KX=1),
    dict(N=1, H=1, W=1, IC=2064, OC=70, KY=1, KX=1),
    dict(N=1, H=33, W=1, IC=80, OC=130, KY=1, KX=1),
    # taps: padding on every side, strides, pixels of one and of five chunks
    dict(N=2, H=5, W=7, IC=16, OC=33, KY=3, KX=3, pads=(1, 1, 1, 1)),
    dict(N=1, H=9, W=6, IC=80, OC=18, KY=3, KX=2, strides=(2, 1), pads=(1, 0, 2, 0)),
    dict(N=3, H=8, W=9, IC=64, OC=48, KY=1, KX=1, strides=(2, 2)),
    dict(N=1, H=6, W=6, IC=256, OC=65, KY=5, KX=5, pads=(2, 2, 2, 2)),
]
SHAPES = ["1,1,1", "1,1,8", "2,1,1", "2,1,4", "2,2,1", "2,2,4", "2,4,1", "4,4,1", "1,1,3"]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("layer", range(len(LAYERS)))
def test_tiles_and_waves(rt, orc, dev, layer, shape):
    rng = np.random.default_rng(seed("direct", layer, shape))
    for kinds, kw in ((("dense", "dense"), dict(mode="LPRELU", zp_in=7)), (("chan16", "chan_odd"), dict(in_u8=False, out_signed=True)),
                      (("window", "window_chan"), dict(zp_in=200, zp_w=131, mode="LRELU"))):
        assert run_views(rt, orc, dev, rng, LAYERS[layer], *kinds, tuning=(("VPX_NCE_DIRECT", shape),), **kw) == "nce_direct"


@pytest.mark.parametrize("family", ["gemm_stride2", "tile", "tile5x5", "stream", "stream_ksplit", "rows16", "rows16_48"])
def test_small_layers_take_it_by_themselves_and_say_so(rt, orc, dev, family):
    g, force, tuning, _ = FAMILIES[family]
    rng = np.random.default_rng(seed("auto", family))
    assert run_views(rt, orc, dev, rng, g, "window_chan", "chan_odd", force=force, tuning=tuning) == "nce_direct"


@pytest.mark.parametrize("family,knob,value", [("stream_ksplit", "VPX_STREAM_KSPLIT", "off"), ("stream", "VPX_CONV_ROWS", 2), ("tile", "VPX_CONV_WAVES", 4),
                                               ("rows16", "VPX_CONV_COLS", 7), ("gemm_stride2", "VPX_GEMM_TILE", 128), ("gemm_stride2", "VPX_GEMM_WAVES", 4)])
def test_a_knob_of_a_family_keeps_its_kernel(rt, orc, dev, family, knob, value):
    g, force, tuning, kernel = FAMILIES[family]
    rng = np.random.default_rng(seed("knob", family))
    assert run_views(rt, orc, dev, rng, g, "dense", "dense", force=force, tuning=tuple(tuning) + ((knob, value),)) == kernel


@pytest.mark.parametrize("family", sorted(FAMILIES))
def test_families_without_it(rt, orc, dev, family):
    g, force, tuning, kernel = FAMILIES[family]
    rng = np.random.default_rng(seed("off", family))
    for in_kind, out_kind, in_u8 in (("dense", "dense", True), ("window_chan", "window", False)):
        assert run_views(rt, orc, dev, rng, g, in_kind, out_kind, in_u8=in_u8, out_signed=not in_u8, force=force,
                         tuning=tuple(tuning) + (("VPX_NCE_DIRECT", "off"),)) == kernel
