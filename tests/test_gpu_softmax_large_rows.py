"""Softmax along the innermost axis of packed fp16 rows, tensors of 2^24 values and more: stores past the caches and, for rows of 129 to 256 values, through them."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width", [(140001, 128 + 1), (66003, 255), (100001, 200), (300007, 60), (200003, 97), (40009, 700), (17001, 1030)])
def test_rows(rt, dev, rows, width):
    import torch
    g = torch.Generator(device="cuda").manual_seed(width)
    x = (torch.randn((rows, width), device=dev, generator=g) * 3).half()
    x[torch.rand((rows, width), device=dev, generator=g) < 0.05] = -65504.0
    whole = torch.full((rows * width + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[:rows * width].view(rows, width)
    rt.softmax(x, y, 1)
    for part, got in zip(x.split(1 << 15), y.split(1 << 15)):
        want = torch.softmax(part.double(), 1)
        # one rounding to fp16 (half of 2^-10 of a value, of 2^-24 below the normal ones); exponents of 40 and less in fp32, 2^-18 of a value
        assert bool(((got.double() - want).abs() <= (2.0 ** -11 + 2.0 ** -17) * want + 2.0 ** -25).all())
    assert bool((whole[rows * width:] == 7).all()), "wrote outside the output"
