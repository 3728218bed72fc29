"""The append of all layers of a captured step in one launch
(pda_rope_append_layers) against one rope_append per layer, bit for bit: one
layer, as many as one launch carries, one more; both layouts, fp16, bf16 and
8-bit K/V; rows outside the arena; arenas of different sizes. And the steps
that must keep their order: layers over one arena, a layer whose input is
another layer's output."""

import pytest
import torch

from instinct_amd import hip_kernels
from instinct_amd.step import DecodeStepGraph

pytestmark = pytest.mark.gpu

PAGE, KV_HEADS, HQ = 16, 2, 6


def arena(gpu, gen, kind, layout, pages, d):
    shape = ((pages, KV_HEADS, PAGE, d) if layout == "pages" else (pages * PAGE, KV_HEADS, d))
    if kind != "int8":
        dtype = torch.bfloat16 if kind == "bf16" else torch.float16
        return tuple(torch.randn(shape, generator=gen, device=gpu).to(dtype) for _ in range(2))
    kv = tuple(torch.randint(-127, 128, shape, generator=gen, device=gpu).to(torch.int8)
               for _ in range(2))
    return kv + tuple(torch.rand(shape[:-1], generator=gen, device=gpu).half() / 40
                      for _ in range(2))


def step_of(gpu, layers, kind="fp16", layout="pages", d=64, batch=5, shared=False):
    gen = torch.Generator(device=gpu).manual_seed(layers)
    width = 4
    # Sequence b's pages; those of the last lie past the smaller arenas' end,
    # so its rows are written in some layers only (and masked in the others).
    seq_tables = torch.arange(batch * width, dtype=torch.int32, device=gpu).view(batch, width)
    arenas = [arena(gpu, gen, kind, layout, batch * width - (width if i % 3 == 2 else 0), d)
              for i in range(1 if shared else layers)]
    arenas = arenas * layers if shared else arenas
    step = DecodeStepGraph(arenas, seq_tables, batch=batch, q_heads=HQ, page_size=PAGE,
                           width=width, scale=d ** -0.5, longest=width * PAGE, dims=d, base=1e6)
    step.slots.copy_(torch.arange(batch, dtype=torch.int32))
    step.positions.copy_(torch.tensor([0, 15, 16, 40, 63][:batch], dtype=torch.int32))
    for group in (step.q, step.k, step.v):
        for t in group:
            t.normal_(generator=gen)
    return step


def one_by_one(step):
    """The step layer by layer on copies of its arenas (a copy per distinct
    arena) and inputs; arenas and outputs."""
    copies = {}
    for a in step.arenas:
        copies.setdefault(a[0].data_ptr(), tuple(t.clone() for t in a))
    arenas = [copies[a[0].data_ptr()] for a in step.arenas]
    tables, lengths, rows = hip_kernels.pack_decode_step(
        step.seq_tables, step.slots, step.positions, width=step.width, page_size=PAGE)
    outs = []
    for i, a in enumerate(arenas):
        scales = a[2:] or None
        q = outs[i - 1] if i and step.q[i] is step.out[i - 1] else step.q[i]
        q = hip_kernels.rope_append(q, step.k[i], step.v[i], a[0], a[1], step.positions, rows,
                                    page_size=PAGE, scales=scales, **step.rope)
        outs.append(hip_kernels.paged_decode_attention(q, a[0], a[1], tables, lengths,
                                                       scales=scales, **step.kw))
    return arenas, outs


def check(step):
    arenas, outs = one_by_one(step)
    step.capture()
    for replay in range(3):
        step.replay()
        torch.cuda.synchronize()
        for layer, (a, want) in enumerate(zip(arenas, outs)):
            assert torch.equal(step.out[layer], want), f"replay {replay} layer {layer}"
            for got, copy in zip(step.arenas[layer], a):
                assert torch.equal(got, copy), f"replay {replay} layer {layer}"
        torch.ones(1 << 18, device=step.positions.device).sum().item()


@pytest.mark.parametrize("layers,kind,layout,d", [
    (1, "fp16", "pages", 64), (48, "fp16", "pages", 64), (49, "fp16", "rows", 96),
    (7, "bf16", "pages", 128), (5, "int8", "pages", 64), (4, "int8", "rows", 80)])
def test_layers_in_one_launch(gpu, layers, kind, layout, d):
    step = step_of(gpu, layers, kind, layout, d)
    assert step._independent()
    check(step)


def test_layers_over_one_arena_keep_their_order(gpu):
    step = step_of(gpu, 3, shared=True)
    assert not step._independent()
    # Every layer overwrites the rows of the one before: only the last layer's
    # stay, while each layer's attention saw its own.
    check(step)


def test_a_layer_fed_by_another_keeps_its_order(gpu):
    step = step_of(gpu, 3)
    step.q[1], step.q[2] = step.out[0], step.out[1]
    assert not step._independent()
    check(step)
