"""MVN with per-channel statistics on NHWC tensors in one launch: channel counts on and off the words, planes that end inside a
row of words, tensors that one workgroup holds and ones that the whole chip does, and the path of a workgroup that does not
meet its partners."""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 8), (2, 3, 3, 1), (3, 7, 5, 3), (8, 8, 8, 16), (1, 18, 10, 51), (5, 33, 31, 17), (2, 37, 55, 16), (2, 64, 64, 64), (1, 100, 101, 20),
          (7, 19, 35, 59), (2, 101, 99, 34), (1, 224, 224, 64), (3, 57, 49, 112), (1, 64, 66, 509), (16, 56, 56, 208), (4, 112, 112, 256), (16, 112, 112, 256),
          (40, 14, 14, 512), (300, 3, 3, 24), (1, 20, 20, 1024)]


def want(x):
    f = x.float()
    mean = f.mean((1, 2), keepdim=True)
    var = (f - mean).square().mean((1, 2), keepdim=True)
    return (f - mean) / (var + 1e-5).sqrt()


def make(dev, shape, offset=0):
    import torch
    n = shape[0] * shape[1] * shape[2] * shape[3]
    g = torch.Generator(device="cuda").manual_seed(n)
    store = torch.empty(n + offset, dtype=torch.float16, device=dev)
    x = store[offset:].view(shape)
    x.copy_(torch.rand(shape, device=dev, generator=g) * 16 - 8 + torch.randn((1, 1, 1, shape[3]), device=dev, generator=g) * 20)
    whole = torch.full((n + offset + 16,), 7.0, dtype=torch.float16, device=dev)
    return x, whole, whole[offset:offset + n].view(shape)


def close(y, w):
    return bool(((y.float() - w).abs() <= 1e-3 * w.abs() + 2e-3).all())


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("offset", [0, 3])
def test_shapes(rt, dev, shape, offset):
    x, whole, y = make(dev, shape, offset)
    rt.mvn(x, y, False, True, 1e-5, "NHWC")
    w = want(x)
    assert close(y, w)
    assert bool((whole[:offset] == 7).all()) and bool((whole[offset + y.numel():] == 7).all()), "wrote outside the output"
    again = x.clone()
    rt.mvn(again, again, False, True, 1e-5, "NHWC")  # in place
    assert close(again, w)


def test_launch_after_launch(rt, dev):
    """Launches of different geometry share the launch counts and the records."""
    import torch
    sets = [make(dev, s) for s in ((1, 224, 224, 64), (2, 101, 99, 34), (16, 56, 56, 208), (2, 37, 55, 16), (4, 112, 112, 256))]
    firsts = []
    for x, _, y in sets:
        rt.mvn(x, y, False, True, 1e-5, "NHWC")
        assert close(y, want(x))
        firsts.append(y.clone())
    for k in range(40):
        x, _, y = sets[(k * 3) % len(sets)]
        y.zero_()
        rt.mvn(x, y, False, True, 1e-5, "NHWC")
        assert torch.equal(y, firsts[(k * 3) % len(sets)])


@pytest.mark.parametrize("shape", [(2, 37, 55, 16), (1, 100, 101, 20), (5, 53, 61, 17), (2, 130, 105, 176), (3, 79, 98, 215), (1, 64, 66, 509), (2, 101, 99, 34), (4, 112, 112, 256),
                                   (16, 112, 112, 256), (1, 448, 448, 256), (1, 900, 900, 17)])
def test_without_waiting(rt, dev, shape):
    import torch
    x, _, y = make(dev, shape)
    rt.mvn(x, y, False, True, 1e-5, "NHWC")
    z = torch.empty_like(y)
    rt.set_tuning("VPX_MVN_FUSED", "nowait")
    try:
        rt.mvn(x, z, False, True, 1e-5, "NHWC")
    finally:
        rt.set_tuning("VPX_MVN_FUSED", None)
    assert torch.equal(y, z)
    rt.mvn(x, z, False, True, 1e-5, "NHWC")
    assert torch.equal(y, z)


def test_in_a_graph(rt, dev):
    import torch
    x, _, y = make(dev, (2, 101, 99, 34))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        rt.mvn(x, y, False, True, 1e-5, "NHWC")
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            rt.mvn(x, y, False, True, 1e-5, "NHWC")
    for k in range(4):
        x.mul_(-1.25)
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert close(y, want(x))


def test_more_workgroups_than_a_launch_holds(rt, dev):
    """65535 images of 128 blocks of 64 channels would be 2^32 lanes in one launch: the three-launch path has them."""
    import torch
    shape = (65535, 2, 1, 8192)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(-2048, 2048, shape, dtype=torch.int16, device=dev, generator=g).half()
    y = torch.full(shape, 7.0, dtype=torch.float16, device=dev)
    rt.mvn(x, y, False, True, 1e-5, "NHWC")
    for n in (0, 1, 32767, 65533, 65534):
        assert close(y[n:n + 1], want(x[n:n + 1]))
    # two values differ from their mean by the same amount: 0 or plus and minus one
    assert bool((y[:, 0].abs() <= 1.001).all()) and torch.equal(y[:, 0], -y[:, 1])
