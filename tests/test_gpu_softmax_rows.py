"""Softmax along the innermost axis of packed fp16 rows of any length at any address: teams of 4 ... 64 lanes, one to four words each."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1, 7, 8, 9, 17, 31, 32, 33, 48, 63, 65, 72, 127, 129, 248, 255, 257, 300, 512, 513, 1023, 1024, 1025, 1535, 1537, 2047, 2048, 2049])
@pytest.mark.parametrize("rows", [1, 65, 1027, 25001])
@pytest.mark.parametrize("offset", [0, 5])
def test_rows(rt, dev, width, rows, offset):
    import torch
    n = rows * width
    g = torch.Generator(device="cuda").manual_seed(n + offset)
    store = torch.empty(n + offset, dtype=torch.float16, device=dev)
    x = store[offset:].view(rows, width)
    x.copy_(torch.randn((rows, width), device=dev, generator=g) * 3)
    x[torch.rand((rows, width), device=dev, generator=g) < 0.05] = -65504.0
    x[rows // 2] = -65504.0  # a row that is masked altogether
    whole = torch.full((n + offset + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[offset:offset + n].view(rows, width)
    rt.softmax(x, y, 1)
    want = torch.softmax(x.double(), 1)
    # one rounding to fp16 (half of 2^-10 of a value, of 2^-24 below the normal ones); exponents of 40 and less in fp32, 2^-18 of a value
    close = lambda got: bool(((got.double() - want).abs() <= (2.0 ** -11 + 2.0 ** -17) * want + 2.0 ** -25).all())
    assert close(y)
    assert bool((whole[:offset] == 7).all()) and bool((whole[offset + n:] == 7).all()), "wrote outside the output"
    rt.softmax(x, x, 1)  # in place
    assert close(x)
