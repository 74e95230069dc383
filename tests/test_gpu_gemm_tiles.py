"""The matmul kernel's tiles (panels of 128 bytes, the last one halved where K is an odd multiple of 64; column sums
shared between the waves of a column) against the oracle, where the panels, the ring of buffers and the tiles end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(rt, orc, dev, rng, M, K, N, tile, in_u8, zp_in, zp_w, out_f16, shift=20, direct="off"):
    import torch
    a = rng.integers(0, 256, (1, M, 1, K), dtype=np.uint8) if in_u8 else rng.integers(-128, 128, (1, M, 1, K)).astype(np.int8)
    b = rng.integers(0, 256, (N, 1, 1, K), dtype=np.uint8) if zp_w else rng.integers(-127, 128, (N, 1, 1, K)).astype(np.int8)
    wt = rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, N), rng.integers(shift, shift + 3, N), rng.integers(-2 ** 15, 2 ** 15, N).astype(np.int32), K)
    lo, hi, zp_out = (-(2 ** 31), 2 ** 31 - 1, 0) if out_f16 else (0, 255, 3)  # (an fp16 output has no zero point)
    want = orc.nce_conv(a, b, wt, orc.ppe(1638, 14, zp_out, lo, hi), zp_in=zp_in, zp_w=zp_w, out_f16=out_f16)
    out = torch.full((1, M, 1, N), 77, dtype=torch.float16 if out_f16 else torch.uint8, device=dev)
    rt.set_tuning("VPX_GEMM_TILE", tile)
    rt.set_tuning("VPX_NCE_DIRECT", direct)
    rt.set_tuning("VPX_GEMM_REGB", "off")
    try:
        rt.nce_task(*(torch.from_numpy(x).to(dev) for x in (a, b, wt)), out, rt.PpeInt(rt.PPE_LPRELU, lo, hi, 1638, 14), zp_in=zp_in, zp_w=zp_w, zp_out=zp_out)
    finally:
        for knob in ("VPX_GEMM_TILE", "VPX_NCE_DIRECT", "VPX_GEMM_REGB"):
            rt.set_tuning(knob, None)
    got = out.cpu().numpy()
    assert np.array_equal(got.view(np.uint16) if out_f16 else got, want), (M, K, N, tile, in_u8, zp_in, zp_w, out_f16)
    return rt.nce_last_kernel()


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448, 512, 576, 704, 1088])
def test_every_end_of_the_panels(rt, orc, dev, tile, K):
    """fewer panels than buffers, one more, half of one; tiles of one row, full, and one past full; rows that start at any byte and
    end in part of a word, also the first of a tile; sums on and off"""
    rng = np.random.default_rng(K + tile)
    for M, N in ((1200, 144), (tile, tile), (tile + 1, 3 * tile + 2), (67, tile + 21), (1000, 49)):
        for in_u8, zp_in in ((True, 128), (True, 7), (False, -5)):
            name = run(rt, orc, dev, rng, M, K, N, tile, in_u8, zp_in, 0, False)
            assert name == "nce_gemm_mfma"


@pytest.mark.parametrize("tile", [None, 64, 128, 256])
@pytest.mark.parametrize("M,K,N", [(1100, 320, 209), (2180, 448, 2070)])
def test_outputs_and_zero_points(rt, orc, dev, tile, M, K, N):
    """fp16 outputs, a weight zero point (the per-row term), scales that clip; more tiles than compute units and fewer"""
    rng = np.random.default_rng(M)
    for in_u8, zp_in, zp_w, out_f16, shift in ((True, 7, 31, False, 20), (False, 3, 0, True, 24), (True, 128, 128, False, 20), (False, 0, 0, False, 9)):
        assert run(rt, orc, dev, rng, M, K, N, tile, in_u8, zp_in, zp_w, out_f16, shift) == "nce_gemm_mfma"


@pytest.mark.parametrize("out_f16", [False, True])
@pytest.mark.parametrize("K", [320, 384, 448, 640, 4096])
def test_large_tiles_fill_the_chip(rt, dev, K, out_f16):
    """342 tiles of 256, more than one for a compute unit, so that panels arrive late and the waves of a tile drift apart: the tables of
    column sums keep to themselves whichever buffer the last panel lies in (bit for bit what tiles of 128 give)"""
    import torch
    M, N = 4600, 4700
    g = torch.Generator(device="cuda").manual_seed(K)
    b = torch.randint(-127, 128, (N, 1, 1, K), dtype=torch.int8, device="cuda", generator=g)
    rng = np.random.default_rng(K)
    wt = torch.from_numpy(rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, N), rng.integers(20, 23, N), rng.integers(-2 ** 15, 2 ** 15, N).astype(np.int32), K)).cuda()
    lo, hi, zp_out = (-(2 ** 31), 2 ** 31 - 1, 0) if out_f16 else (0, 255, 3)
    ppe = rt.PpeInt(rt.PPE_LPRELU, lo, hi, 1638, 14)
    dt = torch.float16 if out_f16 else torch.uint8
    inputs = [torch.randint(0, 256, (1, M, 1, K), dtype=torch.uint8, device="cuda", generator=g) for _ in range(3)]
    outs = {}
    try:
        for tile in (256, 128):
            rt.set_tuning("VPX_GEMM_TILE", tile)
            outs[tile] = [torch.empty((1, M, 1, N), dtype=dt, device="cuda") for _ in inputs]
            for x, out in zip(inputs, outs[tile]):
                rt.nce_task(x, b, wt, out, ppe, zp_in=7, zp_out=zp_out)
            assert rt.nce_last_kernel() == "nce_gemm_mfma"
    finally:
        rt.set_tuning("VPX_GEMM_TILE", None)
    torch.cuda.synchronize()
    for large, small in zip(outs[256], outs[128]):
        assert torch.equal(large, small), (K, out_f16, int((large != small).sum()))
        assert large.unique().numel() > 16


@pytest.mark.parametrize("M,K,N,kernel", [
    (4009, 64, 904, "nce_gemm_mfma"), (6294, 128, 424, "nce_gemm_mfma"), (256, 128, 8848, "nce_gemm_mfma"),  # a short K, tiles of 64 x 64 of the other form
    (294, 384, 5632, "nce_gemm_mfma"), (700, 512, 900, "nce_gemm_mfma"),                                    # 440 and 165 tiles of 64
    (200, 128, 600, "nce_direct"), (100, 512, 500, "nce_direct"), (4, 4096, 1024, "nce_direct"),
])
def test_beside_the_form_that_stages_nothing(rt, orc, dev, M, K, N, kernel):
    assert run(rt, orc, dev, np.random.default_rng(M + N), M, K, N, None, True, 7, 0, False, direct=None) == kernel
