"""MVN over many rows under a shared scale and bias: rows that are no whole words, and what the row kernels keep outside their registers."""
import struct

import pytest


def kernels(path):
    """name -> metadata of every kernel in a library that was built here"""
    msgpack = pytest.importorskip("msgpack")
    blob, out, at = open(path, "rb").read(), {}, 0
    while (at := blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            target = blob[entry + 24:entry + 24 + length]
            entry += 24 + length
            if not size or b"gfx950" not in target:
                continue
            elf = blob[at + offset:at + offset + size]
            sections, = struct.unpack_from("<Q", elf, 40)
            step, count = struct.unpack_from("<HH", elf, 58)
            for i in range(count):
                kind, = struct.unpack_from("<I", elf, sections + i * step + 4)
                note, end = struct.unpack_from("<QQ", elf, sections + i * step + 24)
                end += note
                while kind == 7 and note < end:  # SHT_NOTE
                    name, text, what = struct.unpack_from("<III", elf, note)
                    first = note + 12 + (name + 3) // 4 * 4
                    if what == 32:  # NT_AMDGPU_METADATA
                        out.update({k[".name"]: k for k in msgpack.unpackb(elf[first:first + text]).get("amdhsa.kernels", [])})
                    note = first + (text + 3) // 4 * 4
        at += 24
    return out


def test_row_kernels_keep_nothing_in_scratch(rt):
    rows = {n: k for n, k in kernels(rt.LIB_PATH).items() if "mvn6_rows_kernel" in n}
    assert len(rows) > 50
    assert not [n for n, k in rows.items() if k[".private_segment_fixed_size"]]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [32767, 32771, 65539])
@pytest.mark.parametrize("width,offset", [(768, 1), (1016, 1), (1023, 0), (1025, 0), (1536, 3), (1539, 0), (2047, 0)])
def test_rows_that_are_no_whole_words(rt, dev, rows, width, offset):
    import torch
    n = rows * width
    g = torch.Generator(device="cuda").manual_seed(n)
    store = torch.empty(n + offset, dtype=torch.float16, device=dev)
    x = store[offset:].view(rows, width)
    x.copy_(torch.randn((rows, width), device=dev, generator=g) * 3 + 1)
    scale, bias = (torch.rand((1, width), device=dev, generator=g) + 0.5).half(), torch.randn((1, width), device=dev, generator=g).half()
    whole = torch.full((n + 16,), 7.0, dtype=torch.float16, device=dev)
    y = whole[:n].view(rows, width)
    rt.mvn6(x, y, [1], True, 1e-5, 0, scale, bias)
    for lo in range(0, rows, 1 << 14):
        f = x[lo:lo + (1 << 14)].double()
        f -= f.mean(1, keepdim=True)
        f /= (f.square().mean(1, keepdim=True) + 1e-5).sqrt()
        want = f * scale.double() + bias.double()
        # one rounding to fp16 (half of 2^-10 of a value) and fp32 sums (some 2^-20 of the largest, 8 here)
        assert bool(((y[lo:lo + (1 << 14)].double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -14).all())
    assert bool((whole[n:] == 7).all()), "wrote outside the output"
