"""Prefill chunks whose last position is the last one there is (start + count =
2^31 - 1): the key cursors run past it, and masks are taken next to it. Every
kernel of the dispatch, pages that divide a tile, are divided by it or
neither, key ranges, empty ones among them; against float64. A windowed call
with a table of one page has no usable key and gives zeros."""

import pytest
import torch

from instinct_amd import hip_kernels

pytestmark = pytest.mark.gpu

END = 2**31 - 1
COUNT, WINDOW, HQ = 70, 40, 2


def arenas(gpu, gen, kind, pages, page, d):
    shape = (pages, 1, page, d)
    if kind == "int8":
        k, v = (torch.randint(-127, 128, shape, generator=gen, device=gpu).to(torch.int8)
                for _ in range(2))
        scales = tuple(torch.rand(shape[:-1], generator=gen, device=gpu).half() / 40 + 0.01
                       for _ in range(2))
        return k, v, scales, [(t.half() * s[..., None]).double() for t, s in zip((k, v), scales)]
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    k, v = (torch.randn(shape, generator=gen, device=gpu).to(dtype) for _ in range(2))
    return k, v, None, [k.double(), v.double()]


@pytest.mark.parametrize("page", [1000, 65536])
@pytest.mark.parametrize("splits", [0, 9])
@pytest.mark.parametrize("kind,d", [("fp16", 64), ("bf16", 96), ("fp16", 128), ("bf16", 256),
                                    ("fp16", 512), ("fp16", 80), ("fp16", 81), ("int8", 64)])
def test_last_positions(gpu, kind, d, page, splits):
    gen = torch.Generator(device=gpu).manual_seed(d + page)
    start = END - COUNT
    pages = -(-END // page)
    table = torch.full((pages,), -1, dtype=torch.int32, device=gpu)
    table[-2:] = torch.tensor([1, 0], dtype=torch.int32)
    k, v, scales, dense = arenas(gpu, gen, kind, 2, page, d)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    q = torch.randn((COUNT, HQ, d), generator=gen, device=gpu).to(dtype)
    got = hip_kernels.paged_prefill_attention(q, k, v, table, start=start, page_size=page,
                                              scale=d ** -0.5, window=WINDOW, splits=splits,
                                              scales=scales)
    # Keys start - WINDOW + 1 .. END - 1, from the last two pages.
    rows = [t[[1, 0], 0].reshape(-1, d)[:END - (pages - 2) * page][-(COUNT + WINDOW - 1):]
            for t in dense]
    s = torch.matmul(q.double().transpose(0, 1), rows[0].t().contiguous()) * d ** -0.5
    i = torch.arange(COUNT, device=gpu)[:, None]
    j = torch.arange(COUNT + WINDOW - 1, device=gpu)[None, :]
    s = s.masked_fill((j < i) | (j > i + WINDOW - 1), -torch.inf)
    want = torch.matmul(torch.softmax(s, -1), rows[1].contiguous()).transpose(0, 1)
    # Half an ulp of the weights and of the output, for outputs up to about 4.
    bar = 2 * 4 * 2.0 ** (-8 if kind == "bf16" else -11)
    assert (got.double() - want).abs().max().item() <= bar


@pytest.mark.parametrize("page", [1, 16, 24, 64])
@pytest.mark.parametrize("splits", [0, 9])
@pytest.mark.parametrize("kind,d", [("fp16", 64), ("bf16", 128), ("fp16", 256), ("fp16", 512),
                                    ("fp16", 80), ("int8", 64)])
def test_keys_past_the_table(gpu, kind, d, page, splits):
    gen = torch.Generator(device=gpu).manual_seed(d + page)
    k, v, scales, _ = arenas(gpu, gen, kind, 1, page, d)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    q = torch.randn((COUNT, HQ, d), generator=gen, device=gpu).to(dtype)
    got = hip_kernels.paged_prefill_attention(
        q, k, v, torch.zeros(1, dtype=torch.int32, device=gpu), start=END - COUNT, page_size=page,
        scale=d ** -0.5, window=WINDOW, splits=splits, scales=scales)
    assert not got.any()
