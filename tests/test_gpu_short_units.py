"""Decode calls on both sides of the lines between the one-launch local mode
and the stream, and between the whole-row and the row-sliced merge: the longest
sequence at, one below and one past each line, with shorter ones beside it,
against a float64 reference. Bars: the outputs' half ulp and the weights'
(fp16 2^-11, bf16 2^-8 each, relative to values up to about 4)."""

import pytest
import torch

from instinct_amd import _lib, hip_kernels

PAGE = 16

# q heads, kv heads, head dim, batch, longest, bf16, local mode, merge (1 rows, 2 sliced)
LINES = [
    (14, 2, 64, 1, 511, False, 1, 0), (14, 2, 64, 1, 513, False, 0, 2),
    (14, 2, 64, 32, 768, False, 1, 0), (14, 2, 64, 32, 769, True, 0, 2),
    (28, 4, 128, 1, 320, True, 1, 0), (28, 4, 128, 1, 321, False, 0, 2),
    (28, 4, 128, 16, 512, False, 1, 0), (28, 4, 128, 16, 513, False, 0, 2),
    (32, 8, 128, 2, 640, False, 1, 0), (32, 8, 128, 2, 641, True, 0, 2),
    (32, 8, 128, 8, 768, False, 1, 0), (32, 8, 128, 8, 769, False, 0, 2),
    (8, 4, 256, 1, 256, False, 1, 0), (8, 4, 256, 1, 384, False, 0, 1),
    (32, 8, 96, 2, 768, True, 1, 0), (32, 32, 80, 1, 384, False, 1, 0),
    (32, 32, 80, 1, 385, False, 0, 1), (32, 8, 128, 48, 256, False, 0, 1),
]


@pytest.mark.parametrize("hq,hkv,d,batch,longest,bf16,local,merge", LINES)
def test_rules(hq, hkv, d, batch, longest, bf16, local, merge):
    info = _lib.describe(batch, hq, hkv, d, PAGE, -(-longest // PAGE), longest, 0, bf16=bf16)
    assert (info["local"], info["merge"]) == (local, merge)


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,batch,longest,bf16,local,merge", LINES)
@pytest.mark.parametrize("window", [0, 40])
def test_values(gpu, hq, hkv, d, batch, longest, bf16, local, merge, window):
    gen = torch.Generator(device=gpu).manual_seed(longest + batch)
    dtype = torch.bfloat16 if bf16 else torch.float16
    width = -(-longest // PAGE)
    lengths = torch.randint(0, longest + 1, (batch,), generator=gen, device=gpu).int()
    lengths[0] = longest
    tables = torch.randperm(batch * width, generator=gen, device=gpu).int().view(batch, width)
    draw = lambda *shape: torch.randn(shape, generator=gen, device=gpu).to(dtype)  # noqa: E731
    q, k, v = draw(batch, hq, d), *(draw(batch * width, hkv, PAGE, d) for _ in range(2))
    got = hip_kernels.paged_decode_attention(q, k, v, tables, lengths, page_size=PAGE,
                                             longest=longest, scale=d ** -0.5, window=window)
    eps = 2.0 ** (-8 if bf16 else -11)
    for b, n in enumerate(lengths.tolist()):
        lo = max(0, n - window) if window else 0
        rows = [t[tables[b].long()].transpose(0, 1).reshape(hkv, -1, d)[:, lo:n].double()
                for t in (k, v)]
        if n == 0:
            assert not got[b].any()
            continue
        s = torch.matmul(q[b].double().view(hkv, hq // hkv, d),
                         rows[0].transpose(1, 2).contiguous()) * d ** -0.5
        want = torch.matmul(torch.softmax(s, -1), rows[1].contiguous()).view(hq, d)
        assert (got[b].double() - want).abs().max().item() <= 2 * eps * 4
