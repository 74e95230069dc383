"""Per-channel MVN on NHWC tensors in octets of channels: counts off the octets, whose last octet begins inside the one before, and runs that end
within lines, of a workgroup alone and of ones that exchange sums."""
import pytest

pytestmark = pytest.mark.gpu


# runs of 1, 2, 4 and 8 octets and what is left of them; a position, fewer than the slots of a workgroup, one and several words per lane; units that are
# no multiple of the dies
@pytest.mark.parametrize("channels", [9, 15, 17, 24, 33, 65, 69, 72, 257])
@pytest.mark.parametrize("images,height,width", [(1, 1, 1), (3, 7, 9), (17, 16, 32), (1, 61, 67), (5, 96, 101), (1, 301, 211)])
def test_octets(rt, dev, channels, images, height, width):
    import torch
    shape, n = (images, height, width, channels), images * height * width * channels
    g = torch.Generator(device="cuda").manual_seed(n)
    x = (torch.randn(shape, device=dev, generator=g) * 3 + 1).half()
    whole = torch.full((n + 32,), 7.0, dtype=torch.float16, device=dev)
    y = whole[16:16 + n].view(shape)
    rt.mvn(x, y, False, True, 1e-5, "NHWC")
    f = x.double()
    mean = f.mean((1, 2), keepdim=True)
    want = (f - mean) / ((f - mean).square().mean((1, 2), keepdim=True) + 1e-5).sqrt()
    # one rounding to fp16 (half of 2^-10 of a value) and fp32 sums (some 2^-20 of the largest, 6 here; squares about a first value of up to 5 deviations
    # lose a factor of 26)
    assert bool(((y.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -13).all())
    assert bool((whole[:16] == 7).all()) and bool((whole[16 + n:] == 7).all()), "wrote outside the output"
    first = y.clone()
    rt.set_tuning("VPX_MVN_FUSED", "nowait")
    try:
        rt.mvn(x, y, False, True, 1e-5, "NHWC")
    finally:
        rt.set_tuning("VPX_MVN_FUSED", None)
    assert torch.equal(y, first)
    rt.mvn(x, x, False, True, 1e-5, "NHWC")  # in place
    assert bool(((x.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -13).all())
