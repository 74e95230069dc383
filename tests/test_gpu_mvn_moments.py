"""How exact the variance of MVN over long slices is, where the first words of every slice lie at another level than all others and where not."""
import pytest

pytestmark = pytest.mark.gpu

LANES = 512 * 8  # values of a word for each lane


# words a lane, level of a slice's first four words, of the others
@pytest.mark.parametrize("words,first,others", [(52, 13.7, 0.0), (52, 7.9, 1.1), (52, 5.3, -1.9), (40, 7.9, 0.0), (24, 3.1, 0.3), (8, 6.7, 0.0), (52, 0.0, 0.0), (12, 0.0, 0.0)])
def test_outputs_are_the_nearest(rt, dev, words, first, others):
    import torch
    g = torch.Generator(device="cuda").manual_seed(words)
    x = torch.full((256, words * LANES), others, device=dev)
    x[:, :4 * LANES] = first
    if first == others:
        x += torch.randn(x.shape, device=dev, generator=g)
    else:
        x[:, -LANES:] += torch.randn((256, LANES), device=dev, generator=g) * 2
    x = x.half()
    y = torch.empty_like(x)
    rt.mvn(x.view(1, 1, 256, -1), y.view(1, 1, 256, -1), True, True, 1e-9, "NCHW")
    mean, square = 0.0, 0.0
    for part in x.split(16):
        mean += float(part.double().sum()) / x.numel()
    for part in x.split(16):
        square += float((part.double() - mean).square().sum()) / x.numel()
    z = (x[:, -LANES:].double() - mean) / (square + 1e-9) ** 0.5
    # Half a unit of fp16 is what rounding may be off by.  Some of the thousands of values are near enough to the middle of two for what is more than that to be
    # the error before the rounding.  A lane adds the squares of its words one after another, each addition off by half of 2^-23 of what is there by
    # then, in the mean of all half of the whole: words / 2 of them, eight more inside a word and nine where lanes and slices meet; a deviation has half
    # the error of a variance.  Four roundings more, of the mean, which is no further from zero than the deviation, a difference, a root and a product.
    half_unit = torch.exp2(torch.floor(torch.log2(z.abs())) - 11)
    more = ((y[:, -LANES:].double() - z).abs() - half_unit) / z.abs()
    assert float(more[z.abs() >= 0.5].max()) <= (words / 2 + 17) * 2.0 ** -25 + 8 * 2.0 ** -24


@pytest.mark.parametrize("words", [1, 8, 24, 52])
def test_the_mean_where_the_first_slice_lies_far_off(rt, dev, words):
    """Values next to the mean show how far off it is."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(words)
    x = torch.randn((256, words * LANES), device=dev, generator=g) * 0.02
    x[0] += 8.0
    x = x.half()
    y = torch.empty_like(x)
    rt.mvn(x.view(1, 1, 256, -1), y.view(1, 1, 256, -1), True, True, 1e-9, "NCHW")
    mean = float(x.double().sum()) / x.numel()
    deviation = (float((x.double() - mean).square().sum()) / x.numel() + 1e-9) ** 0.5
    z = (x.double() - mean) / deviation
    near = z.abs() < 2.0 ** -9
    # half a unit of fp16, and the mean: rounded to 2^-24 of itself in three steps (slices, their meeting, the last sum), and slices' means of 2^-24 of a
    # slice's largest in 256 of them, of which the errors of 16 add up
    half_unit = torch.exp2(torch.floor(torch.log2(z.abs())).clamp(min=-14) - 11)
    more = (y.double() - z).abs() - half_unit
    assert int(near.sum()) > 1000
    assert float(more[near].max()) <= (3 * abs(mean) + 0.1 * 16 / 256) * 2.0 ** -24 / deviation + 2.0 ** -33
