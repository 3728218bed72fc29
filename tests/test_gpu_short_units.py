"""Decode calls on both sides of the lines between the one-launch local mode
and the stream, and between the whole-row and the row-sliced merge: the longest
sequence at, one below and one past each line, with shorter ones beside it, over
16-bit and 8-bit K/V, both arena layouts and tables wider than the longest,
against a float64 reference. Bar: the rounding of the outputs and of the weights
(unit roundoff u, fp16 2^-11, bf16 2^-8) reaches 8 u of the outputs' rms where
they lie 4 sigma out; 12 u is asked (8 bits: 24, each element is rounded once
more). At bf16 that is 0.047 of the rms; a page lost of 48 is 0.1 at the rms of
its elements and 0.3 at their largest."""

import pytest
import torch

from instinct_amd import _lib, hip_kernels

PAGE = 16

# q heads, kv heads, head dim, batch, longest, type, local mode, merge (0 none, 1 rows, 2 sliced)
LINES = [
    (14, 2, 64, 1, 511, "fp16", 1, 0), (14, 2, 64, 1, 513, "fp16", 0, 2),
    (14, 2, 64, 32, 768, "fp16", 1, 0), (14, 2, 64, 32, 769, "bf16", 0, 2),
    (28, 4, 128, 1, 320, "bf16", 1, 0), (28, 4, 128, 1, 321, "fp16", 0, 2),
    (28, 4, 128, 16, 512, "fp16", 1, 0), (28, 4, 128, 16, 513, "fp16", 0, 2),
    (32, 8, 128, 2, 640, "fp16", 1, 0), (32, 8, 128, 2, 641, "bf16", 0, 2),
    (32, 8, 128, 8, 768, "fp16", 1, 0), (32, 8, 128, 8, 769, "fp16", 0, 2),
    (8, 4, 256, 1, 256, "fp16", 1, 0), (8, 4, 256, 1, 384, "fp16", 0, 1),
    (32, 8, 96, 2, 768, "bf16", 1, 0), (32, 32, 80, 1, 384, "fp16", 1, 0),
    (32, 32, 80, 1, 385, "fp16", 0, 1), (32, 8, 128, 48, 256, "fp16", 0, 1),
    # 8-bit K/V
    (14, 2, 64, 32, 768, "int8", 1, 0), (14, 2, 64, 32, 769, "int8", 0, 2),
    (28, 4, 128, 1, 320, "int8", 1, 0), (28, 4, 128, 1, 321, "int8", 0, 2),
    (28, 4, 128, 16, 512, "int8", 1, 0), (28, 4, 128, 16, 513, "int8", 0, 2),
    (8, 4, 256, 1, 256, "int8", 1, 0), (8, 4, 256, 1, 257, "int8", 0, 1),
    # The generic kernels above head dim 64: a workgroup per head (without a GPU,
    # as here, 256 of them are taken to be resident), a unit's heads together
    (32, 8, 96, 1, 530, "int8", 1, 0), (32, 8, 96, 1, 531, "int8", 0, 1),
    (32, 32, 80, 1, 350, "int8", 1, 0), (32, 32, 80, 1, 351, "int8", 0, 1),
    (16, 16, 72, 1, 391, "fp16", 1, 0), (16, 16, 72, 1, 392, "fp16", 0, 1),
    (16, 16, 72, 8, 512, "fp16", 1, 0), (16, 16, 72, 8, 513, "fp16", 0, 1),
    (16, 16, 72, 16, 768, "bf16", 1, 0), (16, 4, 96, 16, 640, "int8", 1, 0),
    (24, 8, 112, 1, 366, "fp16", 1, 0), (24, 8, 112, 1, 367, "bf16", 0, 1),
    (64, 8, 112, 1, 666, "fp16", 1, 0), (64, 8, 112, 1, 667, "bf16", 0, 1),
    (16, 8, 112, 10, 400, "fp16", 1, 0), (16, 8, 112, 10, 401, "bf16", 0, 1),
    (16, 8, 72, 10, 768, "bf16", 1, 0), (32, 8, 88, 7, 768, "fp16", 1, 0),
    (16, 8, 112, 10, 640, "int8", 1, 0), (16, 8, 112, 10, 641, "int8", 0, 1),
    (32, 8, 112, 8, 768, "int8", 1, 0),
    (40, 8, 112, 8, 438, "fp16", 1, 0), (40, 8, 112, 8, 439, "bf16", 0, 1),
    (40, 8, 112, 8, 304, "int8", 1, 0), (40, 8, 112, 8, 305, "int8", 0, 1),
    (32, 8, 112, 17, 762, "fp16", 1, 0), (32, 8, 112, 17, 763, "bf16", 0, 1),
    (24, 8, 112, 24, 768, "int8", 1, 0),
    (8, 8, 160, 1, 191, "bf16", 1, 0), (8, 8, 160, 1, 192, "fp16", 0, 1),
    (8, 8, 160, 20, 384, "fp16", 1, 0),
    (8, 2, 200, 16, 256, "int8", 1, 0), (8, 2, 200, 16, 257, "int8", 0, 1),
    (10, 2, 200, 64, 336, "fp16", 1, 0), (10, 2, 200, 64, 337, "fp16", 0, 1),
    (40, 8, 200, 8, 152, "int8", 1, 0), (40, 8, 200, 8, 177, "int8", 0, 1),
    (8, 8, 48, 16, 768, "int8", 1, 0),
]


def choice(hq, hkv, d, batch, longest, kind, page=PAGE, width=0, window=0):
    info = _lib.describe(batch, hq, hkv, d, page, width or -(-longest // page), longest, window,
                         kv_bits=8 if kind == "int8" else 16, bf16=kind == "bf16")
    return info["local"], info["merge"]


@pytest.mark.parametrize("hq,hkv,d,batch,longest,kind,local,merge", LINES)
def test_rules(hq, hkv, d, batch, longest, kind, local, merge):
    assert choice(hq, hkv, d, batch, longest, kind) == (local, merge)


@pytest.mark.parametrize("hq,hkv,d,batch,longest,kind,local,merge", LINES)
def test_rules_over_wider_tables(hq, hkv, d, batch, longest, kind, local, merge):
    """The lines count visible keys: a call at a line stays on its side over a
    wider table, with larger pages, or where a window and not the length ends
    the keys."""
    if local:
        assert choice(hq, hkv, d, batch, longest, kind, width=200)[0] == 1
        assert choice(hq, hkv, d, batch, longest, kind, page=64, width=64)[0] == 1
        assert choice(hq, hkv, d, batch, 4096, kind, width=256, window=longest)[0] == 1


# Generic kernels of which two workgroups share a CU: more heads than CUs, a
# workgroup each.
TWO_TO_A_CU = [
    (8, 8, 112, 40, 320, "fp16", 1, 0), (8, 8, 112, 40, 321, "fp16", 0, 1),
    (8, 8, 112, 48, 768, "bf16", 1, 0), (16, 8, 72, 20, 320, "int8", 1, 0),
    (16, 8, 72, 20, 321, "fp16", 0, 1), (16, 8, 112, 24, 256, "fp16", 1, 0),
    (16, 8, 112, 24, 257, "fp16", 0, 1), (24, 8, 112, 13, 180, "bf16", 1, 0),
    (24, 8, 112, 13, 193, "fp16", 0, 1), (16, 8, 200, 28, 224, "int8", 1, 0),
    (16, 8, 200, 28, 225, "int8", 0, 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,batch,longest,kind,local,merge", TWO_TO_A_CU)
def test_rules_two_to_a_cu(gpu, hq, hkv, d, batch, longest, kind, local, merge):
    assert choice(hq, hkv, d, batch, longest, kind)[0] == local


def test_rules_with_small_pages():
    assert choice(28, 4, 128, 17, 1016, "bf16", page=16, width=64, window=512)[0] == 1
    assert choice(28, 4, 128, 17, 1016, "bf16", page=8, width=127, window=512)[0] == 0


def arena(gpu, gen, kind, layout, pages, hkv, d):
    """K or V of one call: the arena, its scales, and its rows in float64."""
    shape = (pages, hkv, PAGE, d)
    if kind == "int8":
        x = torch.randint(-127, 128, shape, generator=gen, device=gpu).to(torch.int8)
        s = (torch.rand(shape[:-1], generator=gen, device=gpu) * 0.02 + 0.005).half()
        rows = (x.half() * s[..., None]).double()
    else:
        dtype = torch.bfloat16 if kind == "bf16" else torch.float16
        x, s = torch.randn(shape, generator=gen, device=gpu).to(dtype), None
        rows = x.double()
    if layout == "rows":
        x = x.transpose(1, 2).reshape(pages * PAGE, hkv, d).contiguous()
        s = None if s is None else s.transpose(1, 2).reshape(pages * PAGE, hkv).contiguous()
    return x, s, rows


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,batch,longest,kind,local,merge", LINES + TWO_TO_A_CU)
@pytest.mark.parametrize("window,extra,layout", [(0, 0, "pages"), (40, 0, "rows"),
                                                 (0, 50, "rows"), (40, 50, "pages")])
def test_values(gpu, hq, hkv, d, batch, longest, kind, local, merge, window, extra, layout):
    gen = torch.Generator(device=gpu).manual_seed(longest + batch)
    width = -(-longest // PAGE)
    lengths = torch.randint(0, longest + 1, (batch,), generator=gen, device=gpu).int()
    lengths[0] = longest
    tables = torch.randperm(batch * width, generator=gen, device=gpu).int().view(batch, width)
    wide = torch.full((batch, width + extra), -1, dtype=torch.int32, device=gpu)
    wide[:, :width] = tables
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    q = torch.randn((batch, hq, d), generator=gen, device=gpu).to(dtype)
    (k, ks, krows), (v, vs, vrows) = (arena(gpu, gen, kind, layout, batch * width, hkv, d)
                                      for _ in range(2))
    got = hip_kernels.paged_decode_attention(q, k, v, wide, lengths, page_size=PAGE,
                                             longest=longest, scale=d ** -0.5, window=window,
                                             scales=None if ks is None else (ks, vs))
    u = {"bf16": 12 * 2.0 ** -8, "fp16": 12 * 2.0 ** -11, "int8": 24 * 2.0 ** -11}[kind]
    for b, n in enumerate(lengths.tolist()):
        lo = max(0, n - window) if window else 0
        rows = [t[tables[b].long()].transpose(0, 1).reshape(hkv, -1, d)[:, lo:n]
                for t in (krows, vrows)]
        if n == 0:
            assert not got[b].any()
            continue
        s = torch.matmul(q[b].double().view(hkv, hq // hkv, d),
                         rows[0].transpose(1, 2).contiguous()) * d ** -0.5
        want = torch.matmul(torch.softmax(s, -1), rows[1].contiguous()).view(hq, d)
        bar = u * want.square().mean().sqrt().item()
        assert (got[b].double() - want).abs().max().item() <= bar, (b, n)
