"""The pipelined prefill kernels (16-bit K/V at head dims 64, 96, 128, 256)
where they can go wrong, against the float64 prefill oracle: chunks one short
of, at and one past a wave's and a workgroup's queries; keys one short of, at
and one past a tile; page sizes that divide the 64-key tile, are divided by it
or neither; waves whose key range starts or ends inside their workgroup's
(windows, image spans); released pages and keys past the end that hold NaN;
key ranges, empty ones among them; and two query blocks per wave (head dim
128 from 8192 keys on). Bars: the fp16 and bf16 ones of
test_gpu_prefill_shapes."""

import pytest
import torch

from test_gpu_prefill_shapes import case, check

pytestmark = pytest.mark.gpu

# Chunks of a small model: (count, start) around 32, 64 and 128 queries and
# around 64-key tiles.
EDGES = [(1, 0), (31, 33), (32, 32), (33, 95), (63, 0), (64, 64), (65, 127), (127, 1), (128, 0),
         (129, 63), (257, 190)]


@pytest.mark.parametrize("d", [64, 96, 128, 256])
@pytest.mark.parametrize("count,start", EDGES)
def test_edges(gpu, d, count, start):
    page = (16, 24, 5, 64, 128)[(count + d) % 5]
    c = case(gpu, hq=6, hkv=2, d=d, start=start, count=count, page=page, seed=count + d,
             layout=("pages", "rows")[count % 2], bf16=count % 3 == 0)
    check(c, scale=d ** -0.5, what=f"D{d} {count}@{start} page {page}", bf16=count % 3 == 0)


def poison(c, released):
    """NaN in the rows no query may see: released pages and, in the last page,
    the positions past the chunk's end. The table loses the released pages."""
    _, k, v, table = c["t"]
    page, end = c["page"], c["start"] + c["q"].shape[0]
    for i in released:
        p = int(c["table"][i])
        for t in (k, v):
            (t[p] if t.dim() == 4 else t[p * page:(p + 1) * page]).fill_(float("nan"))
        c["table"][i] = -1
        table[i] = -1
    p, used = int(c["table"][-1]), end - (end - 1) // page * page
    for t in (k, v):
        (t[p, :, used:] if t.dim() == 4 else t[p * page + used:(p + 1) * page]).fill_(float("nan"))


@pytest.mark.parametrize("d", [64, 96, 128, 256])
@pytest.mark.parametrize("window,softcap,splits,released,images", [
    (0, 0.0, 0, (1, 2, 9), ()),
    (40, 0.0, 0, (0,), ()),
    (100, 20.0, 3, (), ()),
    (64, 0.0, 0, (), ((150, 90), (330, 17))),
    (0, 0.0, 7, (3,), ((401, 70),)),
    (33, 0.0, 12, (), ()),
])
def test_masks(gpu, d, window, softcap, splits, released, images):
    c = case(gpu, hq=4, hkv=2, d=d, start=139, count=333, seed=d + window + splits,
             layout=("rows", "pages")[d % 3 == 1])
    poison(c, released)
    check(c, scale=d ** -0.5, window=window, softcap=softcap, splits=splits, images=images,
          what=f"D{d} window {window} softcap {softcap} splits {splits} images {images}")


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("count,start,page,window,splits,images", [
    (256, 7936, 16, 0, 0, ()),        # at the line, whole workgroups
    (255, 7937, 24, 0, 1, ()),        # the last wave one query short
    (193, 8001, 16, 0, 0, ()),        # two tiles of 128, the second half a wave
    (1000, 7300, 64, 0, 0, ()),       # eight tiles, ragged
    (256, 8000, 16, 8000, 0, ()),     # the window cuts the first tiles
    (512, 8192, 48, 7900, 5, ((8300, 200),)),
])
def test_two_blocks(gpu, bf16, count, start, page, window, splits, images):
    c = case(gpu, hq=2, hkv=1, d=128, start=start, count=count, page=page, seed=count, bf16=bf16)
    poison(c, ())
    check(c, scale=128 ** -0.5, window=window, splits=splits, images=images, bf16=bf16,
          what=f"{count}@{start} page {page} window {window} splits {splits}")


@pytest.mark.parametrize("d,start", [(64, 300), (128, 300), (128, 8192), (256, 300)])
def test_moving_max(gpu, d, start):
    """Scores that keep growing along the keys, so that the running max moves
    many times and the outputs are rescaled, with far-negative ones between."""
    c = case(gpu, hq=2, hkv=1, d=d, start=start, count=256, seed=d, layout="rows")
    ramp = torch.linspace(0.05, 3.0, c["keys"].shape[0])
    pages = torch.as_tensor(c["table"]).long()
    rows = (pages[:, None] * c["page"] + torch.arange(c["page"])).flatten()
    scale = torch.ones(c["keys"].shape[0])
    scale[rows] = ramp[:len(rows)]
    c["keys"] = (c["keys"] * scale.numpy()[:, None, None]).astype(c["keys"].dtype)
    q, k, v, table = c["t"]
    c["t"] = (q, torch.as_tensor(c["keys"], device=gpu), v, table)
    check(c, scale=4 * d ** -0.5, what=f"D{d} moving max @{start}")


# Calls whose two-block workgroups fill the CUs as well as one-block ones do
# (q heads, count, start, page, window, splits, images), all of one kv head.
TWO_BLOCKS = [
    (64, 256, 7936, 16, 0, 0, ()),               # at the line, whole workgroups
    (64, 255, 7937, 24, 0, 4, ()),               # the last wave one query short
    (64, 193, 8001, 16, 0, 0, ()),               # the second half of 256 a wave and a query
    (16, 1000, 7300, 64, 8300, 0, ()),           # ragged, a window over all keys
    (16, 993, 7300, 5, 0, 8, ((7200, 300), (8100, 150))),
]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("hq,count,start,page,window,splits,images", TWO_BLOCKS)
def test_two_blocks_that_fill_the_cus(gpu, bf16, hq, count, start, page, window, splits, images):
    from instinct_amd.hip_kernels import paged_prefill_attention

    gen = torch.Generator(device=gpu).manual_seed(count)
    dtype = torch.bfloat16 if bf16 else torch.float16
    keys = start + count
    pages = -(-keys // page)
    table = torch.randperm(pages + 3, generator=gen, device=gpu)[:pages].int()
    draw = lambda *shape: torch.randn(shape, generator=gen, device=gpu).to(dtype)  # noqa: E731
    q, k, v = draw(count, hq, 128), draw(pages + 3, 1, page, 128), draw(pages + 3, 1, page, 128)
    scale = 128 ** -0.5
    if count == 193:  # scores that keep growing: the outputs are rescaled many times
        ramp = torch.linspace(0.05, 3.0, pages * page, device=gpu).view(pages, 1, page, 1)
        k[table.long()] = (k[table.long()] * ramp).to(dtype)
        scale *= 4
    released = pages // 2
    table[released] = -1
    got = paged_prefill_attention(q, k, v, table, start=start, page_size=page, scale=scale,
                                  window=window, splits=splits, images=images)
    rows = [t[table.long().clamp(min=0), 0].reshape(-1, 128)[:keys].double() for t in (k, v)]
    pos = start + torch.arange(count, device=gpu)[:, None]
    key = torch.arange(keys, device=gpu)[None, :]
    seen = key <= pos
    for at, length in images:
        seen |= (pos >= at) & (pos < at + length) & (key >= at) & (key < at + length)
    seen &= (key // page) != released
    worst = total = 0.0
    for h in range(hq):
        s = torch.matmul(q[:, h].double(), rows[0].t().contiguous()) * scale
        want = torch.matmul(torch.softmax(s.masked_fill(~seen, -torch.inf), -1), rows[1])
        diff = (got[:, h].double() - want).abs()
        worst, total = max(worst, diff.max().item()), total + diff.mean().item() / hq
    # The bars of the other prefill tests (fp16; bf16: 8 times, the formats' ratio).
    assert worst <= 2e-3 * (8 if bf16 else 1) and total <= 2e-4 * (8 if bf16 else 1)
