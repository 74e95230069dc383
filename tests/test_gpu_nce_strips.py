"""The row-patch convolution with a patch per wave (nce_conv_strips) against the oracle, where its tiles, patches and walks end."""
import numpy as np
import pytest

from test_gpu_nce_views import run_views, seed

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("without_nce_direct")]

LAYERS = [
    # one tile; columns and rows past the image; channels past the last block of 64, not a multiple of 16
    dict(N=1, H=5, W=5, IC=16, OC=33, KY=3, KX=3, pads=(1, 1, 1, 1)),
    dict(N=2, H=30, W=37, IC=16, OC=64, KY=7, KX=7, strides=(2, 2), pads=(3, 3, 3, 3)),
    # more rows under a tile than travel ahead; different strides; K of an odd number of chunks
    dict(N=1, H=41, W=33, IC=16, OC=70, KY=11, KX=3, strides=(2, 1), pads=(1, 0, 5, 4)),
    # rows of more than 64 chunks (60 under 8 columns); six or three chunks a pixel
    dict(N=2, H=9, W=40, IC={8: 96, 16: 96, 32: 48}, OC=48, KY=3, KX=3, pads=(1, 1, 1, 1)),
    # more tiles than waves, one and two blocks of channels; walks of unequal length that cross columns and images
    dict(N=23, H=70, W=129, IC=16, OC=48, KY=2, KX=2),
    dict(N=11, H=64, W=130, IC=32, OC=130, KY=1, KX=3, pads=(1, 1, 0, 0)),
]


@pytest.mark.parametrize("cols", [8, 16, 32])
@pytest.mark.parametrize("layer", range(len(LAYERS)))
def test_tiles_and_walks(rt, orc, dev, layer, cols):
    rng = np.random.default_rng(seed("strips", layer, cols))
    g = dict(LAYERS[layer])
    g["IC"] = g["IC"][cols] if isinstance(g["IC"], dict) else g["IC"]
    tuning = (("VPX_CONV_STRIPS", cols),)
    for kinds, kw in ((("dense", "dense"), dict(mode="LRELU", zp_in=7)), (("chan16", "chan_odd"), dict(in_u8=False, out_signed=True)),
                      (("window", "window_chan"), dict(zp_in=200, zp_w=131, mode="LPRELU"))):
        assert run_views(rt, orc, dev, rng, g, *kinds, tuning=tuning, **kw) == "nce_conv_strips"


@pytest.mark.parametrize("mode,slope", [("NOOP", (1, 0)), ("LRELU", (0, 0)), ("LPRELU", (1638, 14))])
def test_short_ppe_and_the_rule(rt, orc, dev, mode, slope):
    """scales below 1/2 (no clipping), both signs of the multiplier; chosen without a knob from a tile a SIMD on"""
    import torch
    rng = np.random.default_rng(seed("strips ppe", mode))
    N, H, W, IC, OC = 6, 90, 80, 16, 80
    inp, w = rng.integers(0, 256, (N, H, W, IC), dtype=np.uint8), rng.integers(-127, 128, (OC, 5, 5, IC)).astype(np.int8)
    mults = rng.integers(2 ** 13, 2 ** 15, OC) * (rng.choice([-1, 1], OC) if mode != "LRELU" else 1)
    wt = rt.make_weights_table(mults, rng.integers(24, 27, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), 25 * IC)
    want = orc.nce_conv(inp, w, wt, orc.ppe(*slope, 4, 0, 255), zp_in=100, pads=(2, 2, 2, 2))
    out = torch.zeros(want.shape, dtype=torch.uint8, device=dev)
    rt.nce_task(*(torch.from_numpy(a).to(dev) for a in (inp, w, wt)), out, rt.PpeInt(getattr(rt, "PPE_" + mode), 0, 255, 1638, 14), zp_in=100, zp_out=4, pads=(2, 2, 2, 2))
    assert rt.nce_last_kernel() == "nce_conv_strips"
    assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("W", [17, 20, 24, 25, 37, 48])
def test_narrow_planes(rt, dev, W):
    """planes that fall into fewer tiles of 8 columns than of 16, and planes that do not, against the row-patch kernel"""
    import torch
    N, H, IC, OC = 30, 160, 16, 64
    gen = torch.Generator().manual_seed(W)
    inp, w = torch.randint(0, 256, (N, H, W, IC), dtype=torch.uint8, generator=gen).to(dev), torch.randint(-127, 128, (OC, 3, 3, IC), dtype=torch.int8, generator=gen).to(dev)
    rng = np.random.default_rng(W)
    wt = torch.from_numpy(rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, OC), rng.integers(24, 27, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), 9 * IC)).to(dev)
    outs = []
    for knob, kernel in ((None, "nce_conv_strips"), ("off", "nce_conv_rows16")):
        out = torch.zeros((N, H, W, OC), dtype=torch.uint8, device=dev)
        rt.set_tuning("VPX_CONV_STRIPS", knob)
        try:
            rt.nce_task(inp, w, wt, out, rt.PpeInt(rt.PPE_NOOP, 0, 255), zp_in=100, zp_out=4, pads=(1, 1, 1, 1))
        finally:
            rt.set_tuning("VPX_CONV_STRIPS", None)
        assert rt.nce_last_kernel() == kernel
        outs.append(out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("in_u8", [True, False])
@pytest.mark.parametrize("layer", [dict(N=3, H=37, W=70, IC=16, OC=64, KY=7, KX=7, strides=(2, 2), pads=(3, 3, 3, 3)),
                                   dict(N=2, H=70, W=45, IC=32, OC=112, KY=3, KX=3, pads=(1, 1, 1, 1))])
@pytest.mark.parametrize("out_kind", ["dense", "window_chan"])
def test_whole_channels(rt, orc, dev, layer, in_u8, out_kind):
    """patches of up to 14 rows, whole chunks of channels, output rows on words: tiles that end past the image, in a tensor and in a window of one"""
    rng = np.random.default_rng(seed("strips whole", layer["OC"], in_u8, out_kind))
    for mode in ("NOOP", "LPRELU"):
        assert run_views(rt, orc, dev, rng, layer, "dense", out_kind, in_u8=in_u8, out_signed=not in_u8, mode=mode, tuning=(("VPX_CONV_STRIPS", 16),)) == "nce_conv_strips"
