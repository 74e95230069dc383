"""Convolutions as a matmul over (tap, channel) on the matmul kernel's small tiles, against the oracle: every length of a tap from
half a panel on, taps that end inside a panel, padding on every side, strides, one-pixel planes, views, and where the rule takes it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # N, H, W, IC, OC, KY, KX, strides, pads (left, right, top, bottom)
    (2, 9, 11, 64, 70, 3, 3, (1, 1), (1, 1, 1, 1)),      # two taps a panel
    (1, 13, 7, 80, 64, 3, 2, (2, 1), (0, 1, 2, 0)),      # taps of five chunks
    (3, 8, 9, 112, 33, 1, 3, (1, 2), (1, 0, 0, 0)),      # seven
    (1, 20, 20, 128, 65, 5, 5, (1, 2), (2, 2, 2, 2)),    # a panel a tap
    (2, 7, 7, 144, 130, 3, 3, (1, 1), (1, 1, 1, 1)),     # nine; K ends in half a panel
    (5, 5, 6, 208, 17, 3, 3, (2, 2), (1, 1, 1, 1)),
    (1, 1, 1, 272, 48, 3, 3, (1, 1), (1, 1, 1, 1)),      # one pixel: every tap but one outside
    (1, 1, 40, 320, 20, 1, 1, (1, 1), (0, 2, 0, 1)),     # padded 1x1
    (1, 33, 2, 96, 1, 7, 7, (1, 1), (3, 3, 3, 3)),       # windows larger than the plane
    (70, 3, 3, 64, 64, 2, 2, (1, 1), (0, 1, 1, 0)),      # tiles over many images
]


def run(rt, orc, dev, rng, case, tile, zp_in, zp_w, in_u8, out_signed, shift, kernel="gemm", view=False):
    import torch
    N, H, W, IC, OC, KY, KX, strides, pads = case
    x = rng.integers(0, 256, (N, H, W, IC), dtype=np.uint8) if in_u8 else rng.integers(-128, 128, (N, H, W, IC)).astype(np.int8)
    w = rng.integers(0, 256, (OC, KY, KX, IC), dtype=np.uint8) if zp_w else rng.integers(-127, 128, (OC, KY, KX, IC)).astype(np.int8)
    wt = rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, OC), rng.integers(shift, shift + 3, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), KY * KX * IC)
    lo, hi = (-128, 127) if out_signed else (0, 255)
    want = orc.nce_conv(x, w, wt, orc.ppe(1638, 14, 3, lo, hi), zp_in=zp_in, zp_w=zp_w, strides=strides, pads=(pads[2], pads[0], pads[3], pads[1]), out_signed=out_signed)
    dt = torch.int8 if out_signed else torch.uint8
    xd = torch.from_numpy(x).to(dev)
    if view:  # a channel slice and a window of a larger tensor, into a channel slice of one
        big = torch.full((N, H + 2, W + 3, IC + 48), 99, dtype=xd.dtype, device=dev)
        big[:, 1:H + 1, 2:W + 2, 16:16 + IC] = xd
        xd = big[:, 1:H + 1, 2:W + 2, 16:16 + IC]
        whole = torch.full(want.shape[:3] + (OC + 37,), 77, dtype=dt, device=dev)
        out = whole[..., 5:5 + OC]
    else:
        out = torch.full(want.shape, 77, dtype=dt, device=dev)
    for knob, v in (("VPX_CONV_KERNEL", kernel), ("VPX_GEMM_TILE", tile), ("VPX_NCE_DIRECT", "off")):
        rt.set_tuning(knob, v)
    try:
        rt.nce_task(xd, torch.from_numpy(w).to(dev), torch.from_numpy(wt).to(dev), out, rt.PpeInt(rt.PPE_LPRELU, lo, hi, 1638, 14),
                    zp_in=zp_in, zp_w=zp_w, zp_out=3, strides=strides, pads=pads)
    finally:
        for knob in ("VPX_CONV_KERNEL", "VPX_GEMM_TILE", "VPX_NCE_DIRECT"):
            rt.set_tuning(knob, None)
    assert np.array_equal(out.cpu().numpy(), want), (case, tile, zp_in, zp_w, in_u8, out_signed, view, rt.nce_last_kernel())
    if view:
        assert bool((whole[..., :5] == 77).all()) and bool((whole[..., 5 + OC:] == 77).all()), "wrote outside the output"
    return rt.nce_last_kernel()


@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("case", CASES)
def test_taps_and_padding(rt, orc, dev, case, tile):
    rng = np.random.default_rng(case[1] * 31 + case[3])
    for zp_in, zp_w, in_u8, out_signed, shift, view in ((128, 0, True, False, 20, False), (7, 0, True, True, 20, False), (-5, 0, False, False, 12, False),
                                                        (0, 0, False, True, 22, True), (9, 31, True, False, 20, False)):
        assert run(rt, orc, dev, rng, case, tile, zp_in, zp_w, in_u8, out_signed, shift, view=view) == "nce_conv_gemm"


@pytest.mark.parametrize("N,P,C,kernel", [
    (30, 14, 96, "nce_conv_gemm"), (30, 14, 192, "nce_conv_gemm"),  # 92 and 276 tiles of 64
    (16, 30, 160, "nce_conv_gemm"),                                  # 226 tiles of 128
    (2, 30, 128, "nce_conv_tile"),                                   # 58 tiles of 64: a family's
    (40, 8, 256, "nce_conv_stream"), (16, 7, 512, "nce_conv_stream"),  # small planes, K split over waves, in one round
    (40, 7, 512, "nce_conv_gemm"), (32, 7, 384, "nce_conv_gemm"),    # in two rounds; without the split
    (32, 28, 48, "nce_conv_rows16"),                                 # taps of less than half a panel
    (40, 16, 64, "nce_conv_regw"),                                   # 3x3 taps of 64 channels
])
def test_where_the_rule_takes_it(rt, orc, dev, N, P, C, kernel):
    rng = np.random.default_rng(P + C)
    case = (N, P, P, C, C, 3, 3, (1, 1), (1, 1, 1, 1))
    assert run(rt, orc, dev, rng, case, None, 5, 0, True, False, 20, kernel=None) == kernel


@pytest.mark.parametrize("zp,kernel", [(128, "nce_conv_stream"), (5, "nce_conv_gemm")])
def test_small_planes_near_the_direct_form_take_no_scratch(rt, dev, zp, kernel):
    import torch
    g = torch.Generator(device="cuda").manual_seed(zp)
    x = torch.randint(0, 256, (32, 7, 7, 256), dtype=torch.uint8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (256, 3, 3, 256), dtype=torch.int8, device="cuda", generator=g)
    rng = np.random.default_rng(zp)
    wt = torch.from_numpy(rt.make_weights_table(rng.integers(2**14, 2**15, 256), rng.integers(30, 32, 256),
                                                rng.integers(-2**15, 2**15, 256).astype(np.int32), 2304)).cuda()
    out, ref = torch.empty_like(x), torch.empty_like(x)
    ppe = rt.PpeInt(rt.PPE_LRELU, 0, 255, 1, 0)
    rt.nce_task(x, w, wt, out, ppe, zp_in=zp, pads=(1, 1, 1, 1))
    assert rt.nce_last_kernel() == kernel
    rt.set_tuning("VPX_NCE_KERNEL", "naive")
    try:
        rt.nce_task(x, w, wt, ref, ppe, zp_in=zp, pads=(1, 1, 1, 1))
    finally:
        rt.set_tuning("VPX_NCE_KERNEL", None)
    assert torch.equal(out, ref) and ref.unique().numel() > 16


@pytest.mark.parametrize("N,H,W,IC,OC,k,kernel", [
    (10, 34, 218, 224, 64, 3, "nce_conv_gemm"),    # 580 tiles of 128, a round of two a compute unit and some
    (4, 121, 150, 288, 48, 4, "nce_conv_gemm"),    # 576, 568 full
    (27, 43, 137, 288, 64, 3, "nce_direct"),       # 1243, the form that stages nothing on tiles of 64 x 64
    (3, 122, 260, 112, 16, 5, "nce_conv_rows16"),  # K of 2800 whose weights fit LDS beside their rows
    (5, 130, 131, 624, 16, 2, "nce_direct"),       # rows that do not
])
def test_many_tiles_beside_the_gather_kernels(rt, dev, N, H, W, IC, OC, k, kernel):
    """channels that are no multiple of 64 and weights that the row kernels have no room for: which of the forms takes them, and that it agrees with the general kernel"""
    import torch
    g = torch.Generator(device="cuda").manual_seed(IC + k)
    x = torch.randint(0, 256, (N, H, W, IC), dtype=torch.uint8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (OC, k, k, IC), dtype=torch.int8, device="cuda", generator=g)
    rng = np.random.default_rng(IC + k)
    K = k * k * IC
    wt = torch.from_numpy(rt.make_weights_table(rng.integers(2**14, 2**15, OC), rng.integers(30, 32, OC), rng.integers(-2**15, 2**15, OC).astype(np.int32), K)).cuda()
    shape = (N, H + 2 * (k // 2) - k + 1, W + 2 * (k // 2) - k + 1, OC)
    out, ref = (torch.empty(shape, dtype=torch.uint8, device="cuda") for _ in range(2))
    pads = (k // 2,) * 4
    rt.nce_task(x, w, wt, out, rt.PpeInt(rt.PPE_NOOP, 0, 255), zp_in=5, zp_out=128, pads=pads)
    took = rt.nce_last_kernel()
    rt.set_tuning("VPX_NCE_KERNEL", "naive")
    try:
        rt.nce_task(x, w, wt, ref, rt.PpeInt(rt.PPE_NOOP, 0, 255), zp_in=5, zp_out=128, pads=pads)
    finally:
        rt.set_tuning("VPX_NCE_KERNEL", None)
    assert torch.equal(out, ref) and ref.unique().numel() > 16
    assert took == kernel
