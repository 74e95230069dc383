"""Softmax over an outer axis in register slabs: columns of 64, 32 and 16 lanes and every number of waves and of steps the rule
chooses, planes that end in part of a vector and of a tile, against the oracle."""
import numpy as np
import pytest

from test_gpu_sw import _softmax, f16_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("outer,L,inner", [
    (1, 65, 8500), (1, 128, 9001), (2, 256, 5003), (1, 257, 8193), (1, 512, 10001), (1, 513, 9000), (1, 1024, 8321),   # 64 to 140 tiles: 32 lanes
    (1, 70, 8100), (3, 300, 2000), (1, 1000, 4000),                                                                    # fewer: 16 lanes
    (1, 65, 18100), (1, 264, 40003), (1, 320, 18001), (1, 321, 100001), (1, 384, 40001), (1, 385, 18111), (1, 512, 18003),  # more: 64 lanes, 8 waves
    (1, 513, 18001), (1, 768, 18050), (1, 769, 18002),                                                                 # 16 waves
    (1, 67, 30001), (2, 192, 15001), (1, 256, 45001), (1, 383, 30001),                                                 # odd rows, 32 lanes beyond 140 tiles
    (1, 193, 64001), (1, 256, 70001), (1, 385, 60001), (1, 512, 64003), (1, 400, 20002),                               # 16 waves of 13 to 16, 25 to 32 steps
    (1, 129, 100001), (1, 185, 30002), (1, 192, 90001),                                                                # 8 waves of 17 to 24
])
def test_every_shape_of_a_tile(rt, orc, dev, outer, L, inner):
    rng = np.random.default_rng(L + inner)
    x = (rng.standard_normal((outer, L, 1, inner), dtype=np.float32) * 4).astype(np.float16)
    x[0, :, 0, 5] = -np.inf
    x[0, L // 2, 0, 5] = 1.0    # one value among masked ones
    x[-1, :, 0, inner - 1] = 60000.0  # the last column: a partial vector, all equal
    got = _softmax(rt, dev, x.view(np.uint16), 1)
    got = (got if isinstance(got, np.ndarray) else f16_bits(got)).view(np.float16).astype(np.float64).reshape(x.shape)
    e = np.exp(x.astype(np.float64) - x.astype(np.float64).max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    # fp32 arithmetic on the way (sums of L terms, two exponentials, a reciprocal: below 2^-11 together), one rounding to fp16
    assert np.all(np.abs(got - want) <= want * (2.0 ** -11 + 2.0 ** -11) + 2.0 ** -24)
