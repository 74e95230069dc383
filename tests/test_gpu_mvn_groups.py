"""MVN over groups that follow one another in memory (planes of NCHW tensors, whole images), at the edges of its forms: groups
of any length at any address, the ones a workgroup keeps in registers or LDS, and the ones that the whole chip does."""
import pytest

pytestmark = pytest.mark.gpu


def run(rt, dev, shape, across, offset=0):
    import torch
    n = shape[0] * shape[1] * shape[2] * shape[3]
    g = torch.Generator(device="cuda").manual_seed(n + offset)
    store = torch.empty(n + offset, dtype=torch.float16, device=dev)
    x = store[offset:].view(shape)
    x.copy_(torch.rand(shape, device=dev, generator=g) * 16 - 8 + torch.randn((1, shape[1], 1, 1), device=dev, generator=g) * 2)
    whole = torch.full((n + offset + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[offset:offset + n].view(shape)
    rt.mvn(x, y, across, True, 1e-5, "NCHW")
    f = x.float()
    dims = (1, 2, 3) if across else (2, 3)
    mean = f.mean(dims, keepdim=True)
    want = (f - mean) / ((f - mean).square().mean(dims, keepdim=True) + 1e-5).sqrt()
    assert bool(((y.float() - want).abs() <= 1e-3 * want.abs() + 2e-3).all())
    assert bool((whole[:offset] == 7).all()) and bool((whole[offset + n:] == 7).all()), "wrote outside the output"
    again = x.clone()
    rt.mvn(again, again, across, True, 1e-5, "NCHW")  # in place
    assert bool(((again.float() - want).abs() <= 1e-3 * want.abs() + 2e-3).all())
    return x, y


@pytest.mark.parametrize("shape", [(1, 3, 1, 8), (2, 7, 3, 5), (1, 5, 33, 31), (3, 33, 39, 43), (2, 16, 64, 64), (1, 20, 127, 129), (1, 20, 128, 129),
                                   (2, 64, 181, 183), (2, 65, 277, 277), (1, 18, 200, 200), (1, 18, 201, 201), (1, 2, 300, 301), (5, 27, 90, 91)])
@pytest.mark.parametrize("offset", [0, 5])
def test_planes(rt, dev, shape, offset):
    run(rt, dev, shape, False, offset)


@pytest.mark.parametrize("shape", [(1, 3, 7, 11), (3, 5, 63, 65), (16, 7, 49, 51), (17, 7, 49, 51), (1, 64, 257, 255), (2, 31, 201, 203), (4, 256, 64, 64),
                                   (16, 65, 129, 131), (3, 341, 181, 183), (1, 96, 512, 512), (2, 101, 500, 499), (13, 61, 223, 225)])
@pytest.mark.parametrize("offset", [0, 1])
def test_images(rt, dev, shape, offset):
    run(rt, dev, shape, True, offset)


@pytest.mark.parametrize("shape", [(2, 31, 101, 103), (3, 64, 181, 183), (1, 96, 512, 512), (2, 399, 255, 257)])
def test_images_without_waiting(rt, dev, shape):
    import torch
    x, y = run(rt, dev, shape, True)
    z = torch.empty_like(y)
    rt.set_tuning("VPX_MVN_FUSED", "nowait")
    try:
        rt.mvn(x, z, True, True, 1e-5, "NCHW")
    finally:
        rt.set_tuning("VPX_MVN_FUSED", None)
    assert torch.equal(y, z)


# a group per image: 1 ... 16 groups, 2 ... 256 workgroups each
SHAPES = [(1, 3, 64, 65), (16, 7, 49, 51), (3, 5, 63, 65), (1, 64, 257, 255), (1, 1, 65, 64), (2, 31, 201, 203), (7, 3, 50, 50)]


def test_launch_after_launch(rt, dev):
    """Launches of different geometry, waiting or not, share the launch counts and the records."""
    import torch
    sets = [run(rt, dev, s, True) for s in SHAPES]
    for k in range(60):
        x, y = sets[k * 3 % len(sets)]
        z = torch.zeros_like(y)
        rt.set_tuning("VPX_MVN_FUSED", "nowait" if k % 4 == 3 else None)
        try:
            rt.mvn(x, z, True, True, 1e-5, "NCHW")
        finally:
            rt.set_tuning("VPX_MVN_FUSED", None)
        assert torch.equal(z, y), SHAPES[k * 3 % len(sets)]


@pytest.mark.parametrize("shape,across,order", [((4, 256, 64, 64), True, "NCHW"), ((1, 3200, 128, 128), True, "NCHW"), ((1, 448, 448, 256), False, "NHWC"),
                                                ((1, 900, 900, 17), False, "NHWC")])
def test_beside_a_launch_that_holds_compute_units(rt, dev, shape, across, order):
    """With 32 compute units left the workgroups start in eight rounds.  The first one waits 0.5 ms, computes what is missing
    and publishes it; the others find it.  The time is bounded by that and some passes over the tensor (104 MB in 0.4 ms at the
    rate of 32 compute units, both ways), not by a wait and the whole tensor for every workgroup (29 ms)."""
    import time
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    x = (torch.rand(shape, device=dev, generator=g) * 16 - 8).half()
    alone, beside = torch.empty_like(x), torch.empty_like(x)
    src = torch.zeros((65536,), device=dev, dtype=torch.int8)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    sink = torch.empty((cus * 8192,), device=dev, dtype=torch.uint8)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    rt.set_tuning("VPX_CALIB_BLOCKS", str(max(1, cus - 32)))
    try:
        with torch.cuda.stream(a):
            rt.mvn(x, alone, across, True, 1e-5, order)
        rt.calib_mfma_i8(src, sink, 200)
        torch.cuda.synchronize()
        with torch.cuda.stream(b):
            rt.calib_mfma_i8(src, sink, 60000)  # about 26 ms
        time.sleep(0.002)
        with torch.cuda.stream(a):
            start.record()
            rt.mvn(x, beside, across, True, 1e-5, order)
            end.record()
        torch.cuda.synchronize()
    finally:
        rt.set_tuning("VPX_CALIB_BLOCKS", None)
    assert torch.equal(alone, beside)
    print("%s beside a launch on %d of %d compute units: %.3f ms" % (shape, cus - 32, cus, start.elapsed_time(end)))
    assert start.elapsed_time(end) < 4.0
