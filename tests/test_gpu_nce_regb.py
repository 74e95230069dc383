"""The weights-in-registers matmul (nce_gemm_regb) on row lengths that are no multiple of 64 and on blocks of 32, 48 and 64
channels: the end of the last fragment, empty parts of the last block, the last rows."""
import numpy as np
import pytest

from test_gpu_nce_views import run_views, seed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("OC", [16, 32, 48, 80, 96, 144, 208, 256])
@pytest.mark.parametrize("IC", [16, 32, 48, 80, 96, 112, 144, 192, 208, 240])
def test_row_lengths(rt, orc, dev, IC, OC):
    rng = np.random.default_rng(seed("regb", IC, OC))
    g = dict(N=1, H=int(rng.integers(1, 90)), W=7, IC=IC, OC=OC, KY=1, KX=1)
    for kinds, kw in ((("dense", "dense"), dict(mode="LPRELU", zp_in=7)), (("chan16", "chan16"), dict(in_u8=False, out_signed=True, mode="LRELU")),
                      (("dense", "dense"), dict(zp_in=200, zp_w=131, mode="NOOP"))):
        assert run_views(rt, orc, dev, rng, g, *kinds, tuning=(("VPX_GEMM_REGB", "on"),), **kw) == "nce_gemm_regb"


def test_three_fragments_by_size(rt, orc, dev):
    """K = 192, which the dispatch gives it by size alone."""
    rng = np.random.default_rng(seed("regb", 192))
    g = dict(N=1, H=517, W=13, IC=192, OC=144, KY=1, KX=1)
    for kw in (dict(mode="LPRELU", zp_in=7), dict(in_u8=False, out_signed=True, mode="LRELU")):
        assert run_views(rt, orc, dev, rng, g, "dense", "dense", **kw) == "nce_gemm_regb"
