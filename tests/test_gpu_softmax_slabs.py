"""Softmax over an outer axis in register slabs, at the edges of its forms: the counts of steps at which another number of
waves or registers is taken, planes that start off every alignment, runs shorter than a vector, and short packed rows."""
import pytest

pytestmark = pytest.mark.gpu


def check(rt, dev, shape, axis, offset=0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + axis)
    n = 1
    for d in shape:
        n *= d
    store = (torch.randn(n + offset, device=dev, generator=g) * 3).half()
    x = store[offset:].view(shape)
    whole = torch.full((n + offset + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[offset:offset + n].view(shape)
    rt.softmax(x, y, axis)
    want = torch.softmax(x.float(), axis)
    assert bool(((y.float() - want).abs() <= 2e-3 * want + 2.0 ** -24).all())
    assert bool((whole[:offset] == 7).all()) and bool((whole[offset + n:] == 7).all()), "wrote outside the output"
    again = x.clone()
    rt.softmax(again, again, axis)  # in place
    assert torch.equal(again, y)


@pytest.mark.parametrize("steps", [1, 2, 8, 9, 16, 17, 33, 64, 65, 129, 256, 257, 512, 513, 1024])
@pytest.mark.parametrize("inner", [1, 3, 31, 129, 2051])
def test_small(rt, dev, steps, inner):
    check(rt, dev, (2, steps, inner), 1, offset=0 if inner != 129 else 3)


@pytest.mark.parametrize("shape", [(3, 7, 330, 401), (2, 16, 257, 513), (1, 21, 513, 513), (1, 63, 301, 301), (1, 100, 255, 257), (2, 150, 128, 128),
                                   (1, 255, 127, 129), (1, 300, 90, 91), (1, 512, 81, 83), (1, 700, 71, 73)])
def test_large(rt, dev, shape):
    check(rt, dev, shape, 1)


@pytest.mark.parametrize("shape", [(5000, 2, 3), (20000, 8, 5), (3000, 9, 5), (10922, 16, 24), (31837, 17, 31), (700, 40, 7), (8000, 64, 33), (11185, 100, 15),
                                   (90, 300, 3), (1900, 500, 63), (9709, 9, 79), (66052, 2, 127)])
def test_short_runs(rt, dev, shape):
    """Runs shorter than a tile, on either side of the rule between a slab and a lane per line."""
    check(rt, dev, shape, 1)


def test_more_slabs_than_a_launch_holds(rt, dev):
    """2^24 workgroups of four waves are 2^32 lanes."""
    import torch
    shape = (1 << 24, 17, 3)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randint(-9, 10, shape, dtype=torch.int8, device=dev, generator=g).half()
    y = torch.empty_like(x)
    rt.softmax(x, y, 1)
    for part in (slice(0, 1000), slice(1 << 23, (1 << 23) + 1000), slice((1 << 24) - 1000, None)):
        want = torch.softmax(x[part].float(), 1)
        assert bool(((y[part].float() - want).abs() <= 2e-3 * want + 2.0 ** -24).all())
    assert bool(((y.sum(1, dtype=torch.float32) - 1).abs() < 0.01).all())


@pytest.mark.parametrize("rows,length", [(64, 17), (65, 18), (1836, 17), (4096, 33), (12 * 161, 161), (513, 255), (70000, 31)])
def test_short_packed_rows(rt, dev, rows, length):
    check(rt, dev, (rows, length), 1)
