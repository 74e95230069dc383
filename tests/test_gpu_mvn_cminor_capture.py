"""Per-channel MVN on NHWC tensors that one workgroup's registers hold needs nothing but its operands: neither captured on a stream that the
library has not seen nor in place, also where workgroups that exchange sums would be faster."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("shape", [(10, 51, 40, 48), (1, 31, 35, 224), (10, 110, 16, 80), (6, 36, 47, 160), (4, 19, 100, 104), (3, 27, 62, 120)])
def test_captured_without_scratch(rt, dev, shape, inplace):
    import torch
    g = torch.Generator(device="cuda").manual_seed(shape[3])
    x = (torch.randn(shape, device=dev, generator=g) * 3 + 1).half()
    f = x.double()
    mean = f.mean((1, 2), keepdim=True)
    want = (f - mean) / ((f - mean).square().mean((1, 2), keepdim=True) + 1e-5).sqrt()
    a, y = x.clone(), torch.empty_like(x)
    y = a if inplace else y
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    rt.workspace_release(stream=stream)
    refused = []
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            try:
                rt.mvn(a, y, False, True, 1e-5, "NHWC")
            except rt.VpxError as err:
                refused.append(err)
            f.add_(0)  # (the capture is ended normally either way)
    assert not refused, str(refused[0])
    for _ in range(2):
        y.fill_(7)
        a.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        # one rounding to fp16 (half of 2^-10 of a value) and fp32 sums (some 2^-20 of the largest, 6 here; squares about a first value of up to 5
        # deviations lose a factor of 26)
        assert bool(((y.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -13).all())
