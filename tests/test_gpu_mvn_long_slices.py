"""MVN across channels over slices that are summed while they arrive (those for 512 lanes), at the sizes where a lane's words and the
kernel's forms end, over values whose first ones say little about the others."""
import pytest

pytestmark = pytest.mark.gpu

LANES = 512 * 8  # values of a word for each lane


def values(torch, kind, groups, length, dev):
    g = torch.Generator(device="cuda").manual_seed(length)
    x = torch.randn((groups, length), device=dev, generator=g)
    if kind == "far":  # mean 40 times the deviation
        return x * 0.5 + 20
    if kind == "steps":  # runs of ten slices' lengths and less at two levels, little noise: slices that begin at one and go on at the other
        at = torch.arange(length, device=dev) // 70001 % 3
        return x * 0.01 + torch.where(at == 0, 8.0, -3.0)
    return x


@pytest.mark.parametrize("kind", ["plain", "far", "steps"])
@pytest.mark.parametrize("groups,words", [(1, 4.01), (2, 7.98), (1, 8.01), (1, 12), (1, 12.02), (3, 16), (1, 16.03), (1, 20), (2, 23.99), (1, 24.01), (1, 28.01), (1, 32.01), (1, 35.99),
                                          (1, 40), (1, 40.02), (2, 44.01), (1, 48), (2, 51.9)])
def test_long_slices(rt, dev, kind, groups, words):
    import torch
    wpg = 256 // groups
    length = int(words * LANES) // 8 * 8 * wpg - 3
    x = values(torch, kind, groups, length, dev).half().view(groups, 1, 1, length)
    y, z = torch.empty_like(x), torch.empty_like(x)
    rt.mvn(x, y, True, True, 1e-9, "NCHW")
    rt.set_tuning("VPX_MVN_FUSED", "nowait")
    try:
        rt.mvn(x, z, True, True, 1e-9, "NCHW")
    finally:
        rt.set_tuning("VPX_MVN_FUSED", None)
    assert torch.equal(y, z)
    d = x.double()
    d -= d.mean((1, 2, 3), keepdim=True)
    d /= (d.square().mean((1, 2, 3), keepdim=True) + 1e-9).sqrt()
    # half a unit of fp16 (2^-11 of a value, 2^-25 of a subnormal one), and sums of 32 bits: 1e-6 of a deviation, of the mean's 40 as well
    err = (y.double() - d).abs() - d.abs() * (2.0 ** -11 + 1e-5)
    assert float(err.max()) <= 2.0 ** -25 + 5e-5
