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


@pytest.mark.parametrize("shape,depth", [("1,1,1", 8), ("1,1,8", 8), ("2,1,1", 6), ("2,1,8", 6), ("2,2,1", 4), ("2,2,8", 4), ("2,4,1", 3), ("4,4,1", 2)])
@pytest.mark.parametrize("taps", [1, 3])
def test_walks_around_the_steps_asked_for_at_once(rt, orc, dev, shape, depth, taps):
    """K of one step less than a wave asks for, as many, one more, twice as many; taps per step (64 channels) and per lane (48);
    scales below 1/2 (the epilogue without clipping), both signs of the multiplier, odd rows of bytes."""
    import torch
    waves = int(shape.split(",")[2])
    rng = np.random.default_rng(seed("walk", shape, taps))
    for steps in (depth - 1, depth, depth + 1, 2 * depth - 1, 2 * depth):
        for unit in ((64, 48) if taps == 3 else (64,)):
            IC = unit if taps == 3 else 64 * steps * waves
            KY = max(1, steps * waves * 64 // (unit * taps)) if taps == 3 else 1
            N, H, W, OC = 2, KY + 2, 9, 37
            inp = rng.integers(0, 256, (N, H, W, IC), dtype=np.uint8)
            w = rng.integers(-127, 128, (OC, KY, taps, IC)).astype(np.int8)
            mults, shifts = rng.integers(2 ** 13, 2 ** 15, OC) * rng.choice([-1, 1], OC), rng.integers(23, 26, OC)
            wt = rt.make_weights_table(mults, shifts, rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), KY * taps * IC)
            pads = (1, 1, 1, 1) if taps == 3 else (0, 0, 0, 0)
            want = orc.nce_conv(inp, w, wt, orc.ppe(1638, 14, 4, 0, 255), zp_in=101, pads=pads)
            out = torch.zeros(want.shape, dtype=torch.uint8, device=dev)
            rt.set_tuning("VPX_NCE_DIRECT", shape)
            try:
                rt.nce_task(*(torch.from_numpy(a).to(dev) for a in (inp, w, wt)), out, rt.PpeInt(rt.PPE_LPRELU, 0, 255, 1638, 14), zp_in=101, zp_out=4, pads=pads)
            finally:
                rt.set_tuning("VPX_NCE_DIRECT", None)
            assert rt.nce_last_kernel() == "nce_direct"
            assert np.array_equal(out.cpu().numpy(), want), (steps, unit)


@pytest.mark.parametrize("N,H,W,IC,OC,k,s,p,zp", [
    # beside the stream kernel, whose sums of a zero point take scratch: small planes, narrow outputs, inputs that a stride skips lines of
    (54, 5, 5, 512, 176, (3, 3), 1, 1, 5), (17, 6, 6, 512, 400, (3, 3), 1, 1, 5), (86, 4, 26, 768, 128, (2, 2), 2, 0, -3),
    (101, 48, 48, 256, 16, (1, 1), 2, 0, 5), (5, 85, 85, 896, 16, (1, 1), 1, 0, 5), (14, 32, 32, 1664, 64, (1, 3), 2, 0, 5),
    (27, 9, 59, 1664, 109, (1, 3), 3, 0, 5),
    # beside the gather kernel, whose prepared channels do
    (3, 178, 178, 1792, 16, (1, 1), 1, 0, 128), (6, 167, 167, 960, 16, (2, 2), 2, 1, 128), (37, 37, 102, 2048, 16, (1, 1), 2, 0, 5),
    (26, 56, 278, 384, 123, (2, 1), 3, 0, -3),
])
def test_layers_near_the_end_of_its_range_take_no_scratch(rt, dev, N, H, W, IC, OC, k, s, p, zp):
    """captured on a stream that has no scratch block, which a kernel that needs one refuses"""
    import torch
    g = torch.Generator(device="cuda").manual_seed(OC)
    x = torch.randint(0, 256, (N, H, W, IC), dtype=torch.uint8, device="cuda", generator=g)
    if zp < 0:
        x = x.view(torch.int8)
    w = torch.randint(-127, 128, (OC,) + k + (IC,), dtype=torch.int8, device="cuda", generator=g)
    rng = np.random.default_rng(OC)
    K = k[0] * k[1] * IC
    shift = int(round(np.log2(5400.0 * np.sqrt(K) * 24576.0 / 60)))
    wt = torch.from_numpy(rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, OC), rng.integers(shift, shift + 2, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), K)).cuda()
    shape = (N, (H + 2 * p - k[0]) // s + 1, (W + 2 * p - k[1]) // s + 1, OC)
    out, ref = torch.empty(shape, dtype=torch.uint8, device="cuda"), torch.empty(shape, dtype=torch.uint8, device="cuda")
    ppe = rt.PpeInt(rt.PPE_LRELU, 0, 255, 1, 0)

    def layer(y):
        rt.nce_task(x, w, wt, y, ppe, zp_in=zp, strides=(s, s), pads=(p, p, p, p))

    rt.set_tuning("VPX_NCE_KERNEL", "naive")
    try:
        layer(ref)
    finally:
        rt.set_tuning("VPX_NCE_KERNEL", None)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    rt.workspace_release(stream=stream)
    refused = []
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            try:
                layer(out)
            except rt.VpxError as err:
                refused.append(err)
            ref.add_(0)  # (the capture is ended normally either way)
    assert not refused, str(refused[0])
    assert rt.nce_last_kernel() in ("nce_direct", "nce_conv_gemm")
    for _ in range(2):
        out.fill_(77)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and ref.unique().numel() > 16


@pytest.mark.parametrize("N,P,IC,OC,p,kernel", [
    (51, 12, 96, 96, 0, "nce_direct"), (26, 6, 144, 544, 1, "nce_direct"), (14, 15, 144, 144, 1, "nce_direct"),  # taps that end inside a line
    (32, 14, 192, 192, 1, "nce_conv_gemm"), (61, 16, 144, 144, 0, "nce_conv_gemm"),
])
def test_beside_the_matmul_form_of_convolutions(rt, orc, dev, N, P, IC, OC, p, kernel):
    rng = np.random.default_rng(IC + N)
    g = dict(N=N, H=P, W=P, IC=IC, OC=OC, KY=3, KX=3, pads=(p, p, p, p))
    assert run_views(rt, orc, dev, rng, g, "dense", "dense", mode="LRELU", zp_in=5) == kernel
