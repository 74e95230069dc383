"""nce_conv_regb over its whole range of input channels: what it serves is bound by K, the taps times the channels, not by the channels."""
import numpy as np
import pytest

from test_gpu_nce_views import run_views, seed

pytestmark = pytest.mark.gpu

# IC, OC, taps: more than 48 channels under every count of steps, and seven steps for 16 output channels
LAYERS = [(80, 16, (3, 3)), (96, 48, (1, 3)), (80, 16, (2, 2)), (80, 48, (2, 2)), (112, 32, (2, 1)), (176, 48, (1, 2)), (144, 32, (3, 1)), (80, 32, (1, 2)), (368, 16, (1, 2)),
          (272, 16, (3, 1)), (48, 16, (3, 3)), (16, 16, (5, 5)), (16, 32, (5, 5))]


@pytest.mark.parametrize("IC,OC,taps", LAYERS)
def test_blocks_and_taps(rt, orc, dev, IC, OC, taps):
    rng = np.random.default_rng(seed("regb wide", IC, OC, taps))
    for N, H, W, strides, p in ((3, 13, 21, (1, 1), 1), (2, 30, 37, (2, 2), 0)):
        layer = dict(N=N, H=H, W=W, IC=IC, OC=OC, KY=taps[0], KX=taps[1], strides=strides, pads=(p * (taps[1] // 2), p * (taps[1] // 2), p * (taps[0] // 2), p * (taps[0] // 2)))
        for kinds, kw in ((("dense", "dense"), dict(mode="LRELU", zp_in=7)), (("window", "window_chan"), dict(zp_in=200, zp_w=131)), (("chan16", "chan_odd"), dict(in_u8=False, out_signed=True))):
            assert run_views(rt, orc, dev, rng, layer, *kinds, tuning=(("VPX_CONV_KERNEL", "regb"),), **kw) == "nce_conv_regb"


@pytest.mark.parametrize("IC,OC,taps", [(80, 16, (2, 2)), (96, 32, (1, 2)), (176, 16, (1, 2)), (48, 16, (3, 3))])
def test_chosen_where_positions_are_many(rt, orc, dev, IC, OC, taps):
    rng = np.random.default_rng(seed("regb wide rule", IC, OC, taps))
    layer = dict(N=4, H=203, W=301, IC=IC, OC=OC, KY=taps[0], KX=taps[1], strides=(2, 2))
    assert run_views(rt, orc, dev, rng, layer, "dense", "dense", mode="LRELU") == "nce_conv_regb"
