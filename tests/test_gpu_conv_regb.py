"""The convolution with its weights in registers and nothing staged (nce_conv_regb), against the oracle where its blocks, taps and walks end."""
import numpy as np
import pytest

from test_gpu_nce_views import run_views, seed

pytestmark = pytest.mark.gpu

LAYERS = [
    # K of 9 chunks, three steps: less than a block, a last block of one position; rows shorter than a block; images crossed inside one
    dict(N=1, H=3, W=4, IC=16, OC=16, KY=3, KX=3, pads=(1, 1, 1, 1)),
    dict(N=5, H=7, W=7, IC=16, OC=64, KY=3, KX=3, strides=(2, 2), pads=(1, 1, 1, 1)),
    dict(N=1, H=17, W=13, IC=16, OC=32, KY=2, KX=5, strides=(2, 1), pads=(4, 0, 0, 1)),
    # five, seven and thirteen steps; no padding; taps wider than the image
    dict(N=3, H=11, W=33, IC=32, OC=16, KY=3, KX=3),
    dict(N=2, H=21, W=50, IC=32, OC=32, KY=3, KX=3, strides=(1, 2), pads=(1, 1, 1, 1)),
    dict(N=3, H=19, W=19, IC=48, OC=48, KY=3, KX=3, pads=(1, 1, 1, 1)),
    dict(N=2, H=30, W=41, IC=16, OC=32, KY=5, KX=5, strides=(2, 2), pads=(2, 2, 2, 2)),
    dict(N=1, H=5, W=6, IC=16, OC=16, KY=7, KX=7, strides=(2, 2), pads=(3, 3, 3, 3)),
    # several blocks for every wave
    dict(N=9, H=150, W=131, IC=16, OC=16, KY=7, KX=7, strides=(2, 2), pads=(3, 3, 3, 3)),
    dict(N=70, H=61, W=75, IC=16, OC=48, KY=5, KX=3, pads=(1, 1, 2, 2)),
]


@pytest.mark.parametrize("layer", range(len(LAYERS)))
def test_blocks_and_taps(rt, orc, dev, layer):
    rng = np.random.default_rng(seed("conv regb", layer))
    for kinds, kw in ((("dense", "dense"), dict(mode="LRELU", zp_in=7)), (("chan16", "chan_odd"), dict(in_u8=False, out_signed=True)),
                      (("window", "window_chan"), dict(zp_in=200, zp_w=131, mode="LPRELU"))):
        assert run_views(rt, orc, dev, rng, LAYERS[layer], *kinds, tuning=(("VPX_CONV_KERNEL", "regb"),), **kw) == "nce_conv_regb"


@pytest.mark.parametrize("mode,slope", [("NOOP", (1, 0)), ("LRELU", (0, 0)), ("LPRELU", (1638, 14))])
@pytest.mark.parametrize("IC,OC,taps,stride", [(16, 16, 3, 1), (16, 16, 7, 2), (32, 16, 3, 2), (16, 32, 3, 2), (32, 32, 3, 1), (48, 32, 3, 2), (48, 48, 3, 1), (16, 64, 3, 2)])
def test_short_ppe_and_the_rule(rt, orc, dev, mode, slope, IC, OC, taps, stride):
    """scales below 1/2 (no clipping), both signs of the multiplier; chosen without a knob where positions are many"""
    import torch
    rng = np.random.default_rng(seed("conv regb ppe", mode, IC, OC, taps))
    N, H, W = (4, 247, 251) if stride == 1 else (6, 401, 331)
    pad = taps // 2
    inp, w = rng.integers(0, 256, (N, H, W, IC), dtype=np.uint8), rng.integers(-127, 128, (OC, taps, taps, IC)).astype(np.int8)
    mults = rng.integers(2 ** 13, 2 ** 15, OC) * (rng.choice([-1, 1], OC) if mode != "LRELU" else 1)
    wt = rt.make_weights_table(mults, rng.integers(24, 27, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), taps * taps * IC)
    want = orc.nce_conv(inp, w, wt, orc.ppe(*slope, 4, 0, 255), zp_in=100, strides=(stride, stride), pads=(pad, pad, pad, pad))
    out = torch.zeros(want.shape, dtype=torch.uint8, device=dev)
    rt.nce_task(*(torch.from_numpy(a).to(dev) for a in (inp, w, wt)), out, rt.PpeInt(getattr(rt, "PPE_" + mode), 0, 255, 1638, 14), zp_in=100, zp_out=4,
                strides=(stride, stride), pads=(pad, pad, pad, pad))
    assert rt.nce_last_kernel() == "nce_conv_regb"
    assert np.array_equal(out.cpu().numpy(), want)
