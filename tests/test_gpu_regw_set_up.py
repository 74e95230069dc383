"""The weights-in-registers convolution's set-up (channels prepared once, by one wave, beside the staged rows) and the size from
which the dispatcher takes it by itself, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGE = 4096  # output positions x blocks of 64 channels from which the kernel is taken unasked


@pytest.mark.parametrize("N,H,W,OC,strides", [
    (1, EDGE // 64, 64, 64, (1, 1)), (1, EDGE // 64 - 1, 64, 64, (1, 1)),   # the edge, one row short of it
    (3, 27, 26, 70, (1, 1)),                                                # two blocks of channels, the last of six
    (2, 91, 93, 130, (2, 2)),                                               # a stride, three blocks, tiles past the last row
    (7, 25, 24, 16, (1, 1)),                                                # a quarter of the block's channels
    (43, 153, 37, 52, (2, 2)),                                              # tiles of 16 rows, 158.7 KiB of the 159.5 that a workgroup may have
])
@pytest.mark.parametrize("zp,shift,lrelu", [(128, 20, None), (0, 20, (1638, 14)), (7, 12, (1638, 14)), (131, 3, None), (128, 20, (3, 0))])
def test_sizes_around_the_edge(rt, orc, dev, N, H, W, OC, strides, zp, shift, lrelu):
    """sums on and off, the short PPE and the general one (small shifts clip, slopes above 1)"""
    import torch
    rng = np.random.default_rng(N * H + OC + zp)
    inp = rng.integers(0, 256, (N, H, W, 64), dtype=np.uint8)
    w = rng.integers(-127, 128, (OC, 3, 3, 64)).astype(np.int8)
    K = 9 * 64
    wt = rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, OC), rng.integers(shift, shift + 3, OC), rng.integers(-2 ** 15, 2 ** 15, OC).astype(np.int32), K)
    OH, OW = (H - 1) // strides[0] + 1, (W - 1) // strides[1] + 1
    mult, sh = lrelu or (1, 0)
    op = orc.ppe(mult, sh, 3, 0, 255)
    want = orc.nce_conv(inp, w, wt, op, zp_in=zp, strides=strides, pads=(1, 1, 1, 1))
    p = rt.PpeInt(rt.PPE_LPRELU, 0, 255, mult, sh) if lrelu else rt.PpeInt(rt.PPE_NOOP, 0, 255)
    out = torch.zeros((N, OH, OW, OC), dtype=torch.uint8, device=dev)
    for knob in ("off", None):  # (layers of this size the form that stages nothing serves too: asked for, or as the rule has it)
        rt.set_tuning("VPX_NCE_DIRECT", knob)
        out.zero_()
        try:
            rt.nce_task(*(torch.from_numpy(x).to(dev) for x in (inp, w, wt)), out, p, zp_in=zp, zp_out=3, strides=strides, pads=(1, 1, 1, 1))
        finally:
            rt.set_tuning("VPX_NCE_DIRECT", None)
        if knob == "off":
            edge = N * OH * OW * ((OC + 63) // 64) >= EDGE
            assert rt.nce_last_kernel() == ("nce_conv_regw" if edge else "nce_conv_tile")
        assert np.array_equal(out.cpu().numpy(), want), (knob, rt.nce_last_kernel())
