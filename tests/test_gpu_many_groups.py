"""Tensors of so many short groups or rows that one workgroup for every few of them would be more lanes than a launch holds, 2^32.  About 30 GB of device memory."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups,len_", [((1 << 29) + 3, 2), ((1 << 29) + 40, 7), ((1 << 27) + 11, 24), ((1 << 26) + 11, 104)])
def test_groups(rt, dev, groups, len_):
    import torch
    x = torch.empty((groups, len_), dtype=torch.float16, device=dev).normal_(0, 2, generator=torch.Generator(device="cuda").manual_seed(len_))
    y = torch.full_like(x, 70.0)
    rt.mvn(x.view(1, groups, 1, len_), y.view(1, groups, 1, len_), False, True, 1e-3, "NCHW")
    for part, got in zip(x.split(1 << 24), y.split(1 << 24)):
        f = part.float()
        f -= f.mean(1, keepdim=True)
        f /= (f.square().mean(1, keepdim=True) + 1e-3).sqrt()
        # one rounding to fp16 (half of 2^-10 of a value), fp32 on both sides: some 2^-20 of the largest, 5 here
        f -= got
        assert bool((f.abs() <= 2.0 ** -11 * got.float().abs() + 2.0 ** -16).all())
    del x, y, f
    torch.cuda.empty_cache()


def test_a_launch_that_would_be_cut_short_is_refused(rt, dev):
    """rows with gaps between them, two to a wavefront"""
    import torch
    x = torch.zeros((1 << 27, 16), dtype=torch.float16, device=dev)[:, :9]
    with pytest.raises(rt.VpxError, match="launch limit"):
        rt.softmax(x, x, 1, packed=False)
