"""nce_direct with one tile of one block a wave, whose results are read right behind a walk that ends with one product: with and without the
input's zero point to take out, a walk of one step, of the steps asked for at once, one more and of two rounds."""
import numpy as np
import pytest

from test_gpu_nce_views import run_views, seed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["1,1,1", "1,1,4"])
@pytest.mark.parametrize("IC", [16, 64, 512, 576, 1024, 1088])
@pytest.mark.parametrize("in_u8,zp_in", [(True, 128), (True, 7), (False, 0), (False, -5)])
def test_results_behind_one_product(rt, orc, dev, shape, IC, in_u8, zp_in):
    rng = np.random.default_rng(seed("first readers", shape, IC, zp_in))
    for taps, pad, P in ((1, 0, 4), (3, 1, 5)) if IC <= 64 else ((1, 0, 4),):
        layer = dict(N=1, H=P, W=P, IC=IC, OC=16, KY=taps, KX=taps, pads=(pad, pad, pad, pad))
        assert run_views(rt, orc, dev, rng, layer, "dense", "dense", in_u8=in_u8, out_signed=not in_u8, zp_in=zp_in, mode="LRELU",
                         tuning=(("VPX_NCE_DIRECT", shape),)) == "nce_direct"
