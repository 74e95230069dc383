"""The weights-in-registers matmul's set-up: weights dealt out through LDS where one block of channels is all a workgroup has,
channel sums by matrix instructions, rows asked for ahead; against the oracle at every length of K, and where the rule takes it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [16, 64, 80, 112, 128, 144, 192, 208, 240, 256])
@pytest.mark.parametrize("N", [16, 48, 64, 128, 160])
def test_every_length_of_k(rt, orc, dev, K, N):
    """fewer rows than are asked for ahead, and a walk of several row blocks; zero points on (sums) and off (no sums)"""
    import torch
    rng = np.random.default_rng(K * 1000 + N)
    rt.set_tuning("VPX_GEMM_REGB", "on")
    try:
        for M, zp, shift in ((5, 3, 20), (70001 if N * K <= 16384 else 20011, 0, 22), (1000, -77, 12)):
            a, b = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-127, 128, (N, K)).astype(np.int8)
            wt = rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, N), rng.integers(shift, shift + 3, N), rng.integers(-2 ** 15, 2 ** 15, N).astype(np.int32), K)
            want = orc.nce_matmul(a, b, wt, orc.ppe(1638, 14, 0, -128, 127), zp_a=zp)
            out = torch.zeros((M, N), dtype=torch.int8, device=dev)
            rt.nce_matmul(*(torch.from_numpy(x).to(dev) for x in (a, b, wt)), out, rt.PpeInt(rt.PPE_LPRELU, -128, 127, 1638, 14), zp_a=zp)
            assert rt.nce_last_kernel() == "nce_gemm_regb"
            assert np.array_equal(out.cpu().numpy(), want), (M, zp)
    finally:
        rt.set_tuning("VPX_GEMM_REGB", None)


@pytest.mark.parametrize("M,K,N,kernel", [
    (1200, 160, 640, "nce_gemm_regb"), (6000, 160, 640, "nce_gemm_regb"), (3380, 128, 512, "nce_gemm_regb"),  # wide, some blocks of rows a wave
    (5041, 32, 128, "nce_gemm_regb"), (3200, 48, 192, "nce_gemm_regb"), (13146, 128, 48, "nce_gemm_regb"),   # a block for most waves
    (299, 64, 256, "nce_direct"), (529, 256, 64, "nce_direct"),                                             # few rows
    (3417, 256, 512, "nce_gemm_mfma"),                                                                      # the longest K, many channels
])
def test_where_the_rule_takes_it(rt, orc, dev, M, K, N, kernel):
    import torch
    rng = np.random.default_rng(M + N)
    a, b = rng.integers(0, 256, (1, M, 1, K), dtype=np.uint8), rng.integers(-127, 128, (N, 1, 1, K)).astype(np.int8)
    wt = rt.make_weights_table(rng.integers(2 ** 14, 2 ** 15, N), rng.integers(20, 23, N), rng.integers(-2 ** 15, 2 ** 15, N).astype(np.int32), K)
    want = orc.nce_conv(a, b, wt, orc.ppe(1, 0, 128, 0, 255))
    out = torch.zeros((1, M, 1, N), dtype=torch.uint8, device=dev)
    rt.nce_task(*(torch.from_numpy(x).to(dev) for x in (a, b, wt)), out, rt.PpeInt(rt.PPE_NOOP, 0, 255, 1, 0), zp_out=128)
    assert rt.nce_last_kernel() == kernel
    assert np.array_equal(out.cpu().numpy(), want)
