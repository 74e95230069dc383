"""Layer normalisation of contiguous rows: scale and bias asked for beside the row, and teams that walk two or four rows and ask
for the next while they sum one (taken from 8192 rows per team on), against the oracle."""
import numpy as np
import pytest

from test_gpu_sw import _assert_mvn6_close, f16_bits, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width", [
    (1, 8), (3, 1536), (5, 2048), (2, 4096), (2, 4090), (7, 3072),           # one row a team: early and late scale and bias
    (65535, 16), (65537, 24), (131071, 9),                                   # half a wavefront, two rows, four; the last team's rows run out
    (32769, 264), (65541, 320), (32771, 1000), (65539, 768),                 # a wavefront; rows past the last; words that are not whole
])
def test_rows_asked_for_ahead(rt, orc, dev, rows, width):
    import torch
    rng = np.random.default_rng(rows + width)
    x = orc.f32_to_f16((rng.standard_normal((rows, width), dtype=np.float32) * 2 + 0.5))
    sc, bi = orc.f32_to_f16(rng.uniform(0.5, 2, (1, width)).astype(np.float32)), orc.f32_to_f16(rng.normal(0, 1, (1, width)).astype(np.float32))
    xd = to_dev(x, dev, True)
    # (of many rows the first, the last and some between: the oracle walks them one by one)
    pick = np.unique(np.concatenate([np.arange(min(rows, 40)), np.arange(max(0, rows - 40), rows), rng.integers(0, rows, 200)]))
    for s, b in ((sc, bi), (None, bi), (sc, None)):
        out = torch.full_like(xd, 7.0)
        rt.mvn6(xd, out, [1], True, 1e-5, 0, None if s is None else to_dev(s, dev, True), None if b is None else to_dev(b, dev, True))
        got = f16_bits(out)
        _assert_mvn6_close(got[pick], orc.mvn6_f16(np.ascontiguousarray(x[pick]), [1], True, 1e-5, 0, s, b), orc, "%d x %d" % (rows, width))
        # every other row by a second calculation: no row of unit-variance output is left as it was
        y = out.float()
        if s is not None and b is None:
            y = y / to_dev(s, dev, True).float()
            assert float(y.mean(1).abs().max()) < 0.02 and (width < 16 or float((y.var(1, unbiased=False) - 1).abs().max()) < 0.02)
