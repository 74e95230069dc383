"""MVN over short groups and few rows, where its forms meet: runs of groups through LDS, a group per team of lanes in registers, a row
for 512 lanes of a workgroup."""
import pytest

from test_gpu_mvn_groups import run

pytestmark = pytest.mark.gpu


# (groups, values of a group): under eight values; either side of 8192 groups, 16384, 2^18; whole words and not; the longest of each form
@pytest.mark.parametrize("groups,len_", [(64, 1), (65, 7), (512, 3), (16383, 5), (16385, 7), (63, 9), (64, 8), (8192, 9), (8193, 9), (8193, 16), (16400, 63),
                                         (9000, 65), (9001, 128), (9000, 129), (8200, 511), (8200, 512), (8200, 513), (1024, 1023), (262143, 70), (262145, 70)])
def test_groups(rt, dev, groups, len_):
    run(rt, dev, (1, groups, 1, len_), False)


@pytest.mark.parametrize("rows", [1, 256, 257])
@pytest.mark.parametrize("width", [641, 648, 2049, 4096, 4097, 8192, 8193, 12288, 12290, 16384])
@pytest.mark.parametrize("affine", [False, True])
def test_rows(rt, dev, rows, width, affine):
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows * width)
    x = (torch.randn((rows, width), device=dev, generator=g) * 3 + 1).half()
    scale, bias = (torch.rand((1, width), device=dev, generator=g) + 0.5).half(), torch.randn((1, width), device=dev, generator=g).half()
    whole = torch.full((rows * width + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[:rows * width].view(rows, width)
    rt.mvn6(x, y, [1], True, 1e-5, 0, *((scale, bias) if affine else (None, None)))
    f = x.double()
    mean = f.mean(1, keepdim=True)
    want = (f - mean) / ((f - mean).square().mean(1, keepdim=True) + 1e-5).sqrt()
    if affine:
        want = want * scale.double() + bias.double()
    # one rounding to fp16 (half of 2^-10 of a value) and fp32 sums (some 2^-20 of the largest, 6 here)
    assert bool(((y.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -14).all())
    assert bool((whole[rows * width:] == 7).all()), "wrote outside the output"
