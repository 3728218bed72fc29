"""The calls this library is used for, to be timed and checked.

A serving engine calls the library in three ways: one decode attention per
layer and step over all running sequences, one prefill attention per layer and
prompt chunk, and, where it captures its steps, a whole decode step (packing,
RoPE + K/V append and decode attention of every layer) as one graph. The cases
take the head shapes, lengths, layouts and element types of the repository's
own configurations and tests, from one short sequence to a full batch.

Lengths belong to a case (a seed of their own draws them), so that its work is
known; page tables and all values come from the seed of the preparation.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT / "llm-inference_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "llm-inference_amd"))

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "int8": torch.float16}


def _decode(name, heads, *, batch, low, high, spread="uniform", dtype="fp16", layout="pages",
            page=16, window=0, softcap=0.0, shared=0, prefix=0, lengths_seed=1):
    q_heads, kv_heads, head_dim = heads
    case = dict(kind="decode", q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, batch=batch,
                low=low, high=high, spread=spread, dtype=dtype, layout=layout, page=page,
                window=window, softcap=softcap, shared=shared, prefix=prefix,
                lengths_seed=lengths_seed)
    return dict(case, name=name) if name else case


def _prefill(name, heads, *, start, count, dtype="fp16", layout="pages", page=16, window=0,
             softcap=0.0):
    q_heads, kv_heads, head_dim = heads
    case = dict(kind="prefill", q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                start=start, count=count, dtype=dtype, layout=layout, page=page, window=window,
                softcap=softcap)
    return dict(case, name=name) if name else case


def _step(name, heads, *, layers, batch, low, high, dtype="fp16", page=16, lengths_seed=1):
    q_heads, kv_heads, head_dim = heads
    case = dict(kind="step", q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, layers=layers,
                batch=batch, low=low, high=high, spread="uniform", dtype=dtype, page=page,
                window=0, shared=0, prefix=0, lengths_seed=lengths_seed)
    return dict(case, name=name) if name else case


def listed():
    return [
        # One user early in a chat: the smallest call, all latency.
        _decode("decode-one-short", (28, 4, 128), batch=1, low=777, high=777, dtype="bf16"),
        # A full batch of mixed contexts on a 7B shape: the headline decode call.
        _decode("decode-batch64", (28, 4, 128), batch=64, low=512, high=8192, lengths_seed=2),
        # The same batch over an 8-bit cache.
        _decode("decode-batch64-int8", (28, 4, 128), batch=64, low=512, high=8192, dtype="int8",
                lengths_seed=2),
        # One user with a long document: a single sequence spread over the GPU.
        _decode("decode-long", (32, 8, 128), batch=1, low=32768, high=32768),
        # A sliding-window layer of a batch deep in its contexts.
        _decode("decode-window", (8, 4, 256), batch=32, low=4096, high=32768, window=1024,
                lengths_seed=4),
        # Continuous batching at its largest: contexts from 16 to 64K tokens, a
        # quarter of the sequences on one shared prefix.
        _decode("decode-mix256", (32, 8, 128), batch=256, low=16, high=65536, spread="log",
                shared=64, prefix=2048, lengths_seed=5),
        # A global layer with 512-wide heads at the longest context, bf16.
        _decode("decode-global-d512", (16, 2, 512), batch=1, low=261840, high=261840,
                dtype="bf16"),
        # A fresh prompt on the 7B shape.
        _prefill("prefill-prompt", (28, 4, 128), start=0, count=4096),
        # The last chunk of a long prompt, as the scheduler cuts it, bf16.
        _prefill("prefill-long-chunk", (28, 4, 128), start=32256, count=512, dtype="bf16"),
        # A prompt of odd length after a short cached prefix on a small model,
        # over the reference's row arena.
        _prefill("prefill-ragged-d64", (14, 2, 64), start=389, count=1531, layout="rows"),
        # A burst chunk in a sliding-window layer with 256-wide heads, bf16.
        _prefill("prefill-window-d256", (16, 8, 256), start=6144, count=2048, dtype="bf16",
                 window=1024),
        # A whole captured decode step of a small model: 24 layers in one graph.
        _step("step-graph", (14, 2, 64), layers=24, batch=8, low=1024, high=1024),
    ]


HEADS = [(14, 2, 64), (16, 16, 64), (32, 32, 80), (32, 8, 96), (28, 4, 128), (32, 8, 128),
         (40, 8, 128), (8, 4, 256), (16, 8, 256), (16, 2, 512)]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Any of the three uses, over the declared ranges; bounded so that no
    drawn case reads more K/V than the mixed batch nor takes longer."""
    heads = rng.choice(HEADS)
    q_heads, kv_heads, head_dim = heads
    dtype = rng.choice(["fp16", "bf16", "int8"])
    layout = rng.choice(["pages", "pages", "rows"])
    page = rng.choice([16, 16, 16, 32, 64])
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "step"])
    if kind == "step":
        batch = _log(rng, 1, 64)
        high = _log(rng, 64, 4096)
        layers = rng.randint(4, 24)
        while layers * batch * high * kv_heads * head_dim * 4 > 4e9:
            high = max(64, high // 2)
        return _step(None, heads, layers=layers, batch=batch, low=max(1, high // rng.randint(1, 8)),
                     high=high, dtype="fp16" if dtype == "int8" else dtype, page=page,
                     lengths_seed=rng.randrange(1 << 20))
    window = rng.choice([0, 0, 0, 512, 1024, 4096])
    softcap = rng.choice([0.0, 0.0, 0.0, 50.0])
    if kind == "decode":
        batch = _log(rng, 1, 256)
        high = _log(rng, 64, 65536)
        while batch * min(high, window or high) * kv_heads * head_dim * 4 > 8e9:
            high = max(64, high // 2)
        return _decode(None, heads, batch=batch, low=max(1, high // rng.randint(1, 16)), high=high,
                       dtype=dtype, layout=layout, page=page, window=window, softcap=softcap,
                       lengths_seed=rng.randrange(1 << 20))
    count = _log(rng, 16, 4096)
    start = rng.choice([0, _log(rng, 16, 65536)])
    # At most the multiplications of an 8K-token prompt on the 7B shape.
    while 4 * head_dim * q_heads * count * (start + count) > 1e12:
        start //= 2
        count = max(16, count // 2 + 1) if start < count else count
    return _prefill(None, heads, start=start, count=count, dtype=dtype, layout=layout, page=page,
                    window=window, softcap=softcap)


def _lengths(case):
    """Lengths of a decode batch and which of its sequences share the prefix."""
    rng = np.random.default_rng(case["lengths_seed"])
    low, high, batch = case["low"], case["high"], case["batch"]
    if case["spread"] == "log":
        n = np.floor(np.exp(rng.uniform(math.log(low), math.log(high), batch))).astype(np.int64)
    else:
        n = rng.integers(low, high + 1, batch)
    n = np.clip(n, low, high)
    sharers = np.zeros(batch, dtype=bool)
    if case["shared"]:
        sharers[rng.choice(batch, size=case["shared"], replace=False)] = True
        k = int(sharers.sum())
        n[sharers] = np.floor(np.exp(rng.uniform(math.log(case["prefix"] + 1), math.log(high),
                                                 k))).astype(np.int64)
        n[sharers] = np.clip(n[sharers], case["prefix"] + 1, high)
    return n, sharers


def _tables(case, rng, lengths, sharers):
    """Page lists over a permuted arena (shared prefixes on the same pages, the
    pages before a window released), packed with zeros, and the arena's pages."""
    page, window = case["page"], case["window"]
    width = -(-int(lengths.max()) // page)
    prefix = case["prefix"] // page if case["shared"] else 0
    packed = np.zeros((len(lengths), width), dtype=np.int32)
    spans = []
    for b, n in enumerate(lengths):
        begin = max(0, int(n) - window) // page if window else 0
        packed[b, :begin] = -1
        if sharers[b]:
            packed[b, :prefix] = np.arange(prefix)
            begin = prefix
        spans.append((begin, -(-int(n) // page)))
    need = sum(e - s for s, e in spans)
    order = prefix + rng.permutation(need)
    at = 0
    for b, (s, e) in enumerate(spans):
        packed[b, s:e] = order[at:at + e - s]
        at += e - s
    return packed, prefix + need


def _normal(gen, shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=gen)


def _arena(case, gen, pages, dtype):
    """Keys and values (and their scales for an 8-bit cache) of one layer."""
    page, heads, dim = case["page"], case["kv_heads"], case["head_dim"]
    rows = case.get("layout", "pages") == "rows"
    shape = (pages * page, heads, dim) if rows else (pages, heads, page, dim)
    if case["dtype"] != "int8":
        return (_normal(gen, shape, dtype), _normal(gen, shape, dtype)), None
    # Rows of a quantized N(0, 1): integers over the int8 range, each row's
    # scale its largest magnitude over 127 (2.5 to 3.5 for N(0, 1) rows).
    kv = [torch.empty(shape, dtype=torch.int8, device="cuda") for _ in range(2)]
    for t in kv:
        flat = t.view(-1)
        block = 1 << 28
        for s in range(0, flat.numel(), block):
            part = torch.empty(min(block, flat.numel() - s), dtype=torch.float16, device="cuda")
            flat[s:s + block] = part.normal_(0.0, 42.0, generator=gen).clamp_(-127, 127).round_()
    scales = tuple(torch.empty(shape[:-1], dtype=torch.float16, device="cuda")
                   .uniform_(2.5 / 127, 3.5 / 127, generator=gen) for _ in range(2))
    return tuple(kv), scales


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    scale = case["head_dim"] ** -0.5
    dim, q_heads, kv_heads = case["head_dim"], case["q_heads"], case["kv_heads"]
    if case["kind"] == "prefill":
        end = case["start"] + case["count"]
        need = -(-end // case["page"])
        table = rng.permutation(need).astype(np.int32)
        if case["window"]:
            table[:max(0, case["start"] - case["window"] + 1) // case["page"]] = -1
        kv, scales = _arena(case, gen, need, dtype)
        return dict(case=case, kv=kv, scales=scales, scale=scale,
                    table=torch.as_tensor(table, device="cuda"),
                    q=_normal(gen, (case["count"], q_heads, dim), dtype))
    lengths, sharers = _lengths(case)
    packed, pages = _tables(case, rng, lengths, sharers)
    if case["kind"] == "decode":
        kv, scales = _arena(case, gen, pages, dtype)
        return dict(case=case, kv=kv, scales=scales, scale=scale, longest=int(lengths.max()),
                    tables=torch.as_tensor(packed, device="cuda"),
                    lengths=torch.as_tensor(lengths.astype(np.int32), device="cuda"),
                    q=_normal(gen, (case["batch"], q_heads, dim), dtype))
    from instinct_amd.step import DecodeStepGraph

    layers = case["layers"]
    kv = _normal(gen, (layers, 2, pages, kv_heads, case["page"], dim), dtype)
    graph = DecodeStepGraph([(kv[i, 0], kv[i, 1]) for i in range(layers)],
                            torch.as_tensor(packed, device="cuda"), batch=case["batch"],
                            q_heads=q_heads, page_size=case["page"], width=packed.shape[1],
                            scale=scale, longest=int(lengths.max()), dims=dim, base=1e6)
    graph.slots.copy_(torch.arange(case["batch"], dtype=torch.int32))
    graph.positions.copy_(torch.as_tensor((lengths - 1).astype(np.int32)))
    for group in (graph.q, graph.k, graph.v):
        for t in group:
            t.normal_(generator=gen)
    graph.capture()
    return dict(case=case, kv=kv, graph=graph)


def run(state):
    from instinct_amd.hip_kernels import paged_decode_attention, paged_prefill_attention

    case = state["case"]
    if case["kind"] == "decode":
        return paged_decode_attention(state["q"], *state["kv"], state["tables"], state["lengths"],
                                      page_size=case["page"], longest=state["longest"],
                                      scale=state["scale"], window=case["window"],
                                      softcap=case["softcap"], scales=state["scales"])
    if case["kind"] == "prefill":
        return paged_prefill_attention(state["q"], *state["kv"], state["table"],
                                       start=case["start"], page_size=case["page"],
                                       scale=state["scale"], window=case["window"],
                                       softcap=case["softcap"], scales=state["scales"])
    state["graph"].replay()
    return {"out": state["graph"].out, "kv": state["kv"]}


def _seen(case):
    """Keys each query of a prefill chunk sees."""
    n = case["start"] + 1 + np.arange(case["count"], dtype=np.int64)
    return np.minimum(n, case["window"]) if case["window"] else n


def work(case):
    dim, q_heads, kv_heads = case["head_dim"], case["q_heads"], case["kv_heads"]
    row = kv_heads * (dim * 2 if case["dtype"] != "int8" else dim + 2) * 2  # K and V of one token
    if case["kind"] == "prefill":
        seen = _seen(case)
        keys = min(case["start"] + case["count"], case["window"] + case["count"] - 1
                   if case["window"] else 1 << 62)
        return {"bytes": keys * row + 2 * case["count"] * q_heads * dim * 2
                + 4 * -(-keys // case["page"]),
                "flops": 4 * dim * q_heads * int(seen.sum())}
    lengths, sharers = _lengths(case)
    spans = np.minimum(lengths, case["window"]) if case["window"] else lengths
    unique = int(spans.sum())
    if case["shared"]:
        unique -= (int(sharers.sum()) - 1) * case["prefix"]
    layers = case.get("layers", 1)
    tokens = case["batch"] * dim * 2
    cost = layers * (unique * row + 2 * tokens * q_heads)
    if case["kind"] == "step":
        cost += layers * 2 * 2 * tokens * kv_heads  # the new rows in and out
    tables = 4 * int((-(-spans // case["page"])).sum()) + 4 * case["batch"]
    return {"bytes": cost + tables, "flops": layers * 4 * dim * q_heads * int(spans.sum())}


def tolerance(case):
    """Probabilities and outputs are rounded to the 16-bit type: two roundings
    of half an ulp, the first averaged over the keys. Four times the error
    seen against 64 bits (fp16 and int8 3.6e-4, bf16 2.4e-3)."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3}


def _softcap(s, cap):
    return cap * torch.tanh(s / cap) if cap > 0 else s


def _rows(state, pages, lo, hi):
    """Keys and values of positions lo .. hi - 1 in float64, [n, kv heads, D]."""
    page = state["case"]["page"]
    pos = torch.arange(lo, hi, device="cuda")
    ids = pages[(pos // page).long()].long()
    got = []
    for j in range(2):
        t = state["kv"][j]
        x = t[ids * page + pos % page] if t.dim() == 3 else t[ids, :, pos % page]
        x = x.double()
        if state["scales"] is not None:
            s = state["scales"][j]
            s = s[ids * page + pos % page] if s.dim() == 2 else s[ids, :, pos % page]
            x = x * s.double()[..., None]
        got.append(x)
    return got


def _decode_exact(state, lengths):
    case = state["case"]
    window, group = case["window"], case["q_heads"] // case["kv_heads"]
    out = torch.zeros((case["batch"], case["q_heads"], case["head_dim"]), dtype=torch.float64,
                      device="cuda")
    for b, n in enumerate(lengths):
        q = state["q"][b].double().view(case["kv_heads"], group, -1)
        lo = max(0, int(n) - window) if window else 0
        k, v = _rows(state, state["tables"][b], lo, int(n))
        s = torch.matmul(q, k.permute(1, 2, 0).contiguous()) * state["scale"]
        p = torch.softmax(_softcap(s, case.get("softcap", 0.0)), dim=-1)
        out[b] = torch.matmul(p, v.transpose(0, 1).contiguous()).view(case["q_heads"], -1)
    return out


def _prefill_exact(state):
    case = state["case"]
    start, count, window = case["start"], case["count"], case["window"]
    group = case["q_heads"] // case["kv_heads"]
    out = torch.empty((count, case["q_heads"], case["head_dim"]), dtype=torch.float64,
                      device="cuda")
    for q0 in range(0, count, 512):
        q1 = min(q0 + 512, count)
        lo = max(0, start + q0 - window + 1) if window else 0
        k, v = _rows(state, state["table"], lo, start + q1)
        at = start + torch.arange(q0, q1, device="cuda")[:, None]
        key = torch.arange(lo, start + q1, device="cuda")[None]
        hidden = (key > at) | (key <= at - window) if window else key > at
        for h in range(case["q_heads"]):
            s = state["q"][q0:q1, h].double() @ k[:, h // group].t().contiguous()
            s = _softcap(s * state["scale"], case["softcap"]).masked_fill_(hidden, -math.inf)
            out[q0:q1, h] = torch.softmax(s, dim=-1) @ v[:, h // group].contiguous()
    return out


def _rotate(x, positions, base):
    """RoPE of [n, heads, D] in float64; angles are the float32 products the
    call is defined on (position times inverse frequency)."""
    half = x.shape[-1] // 2
    power = (-np.arange(half, dtype=np.float32) * np.float32(2)) / np.float32(x.shape[-1])
    freq = np.power(np.float32(base), power, dtype=np.float32)
    angle = torch.as_tensor(positions.astype(np.float32)[:, None] * freq, device="cuda").double()
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half].double(), x[..., half:].double()
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "prefill":
        return _prefill_exact(state)
    lengths, _ = _lengths(case)
    if case["kind"] == "decode":
        return _decode_exact(state, lengths)
    graph, page = state["graph"], case["page"]
    outs, kv = [], state["kv"].double()
    at = torch.as_tensor(lengths - 1, device="cuda")
    ids = graph.seq_tables[torch.arange(case["batch"], device="cuda"), (at // page).long()].long()
    for layer in range(case["layers"]):
        kv[layer, 0][ids, :, (at % page).long()] = _rotate(graph.k[layer], lengths - 1, 1e6)
        kv[layer, 1][ids, :, (at % page).long()] = graph.v[layer].double()
        one = dict(case=case, kv=(kv[layer, 0], kv[layer, 1]), scales=None,
                   tables=graph.seq_tables, scale=case["head_dim"] ** -0.5,
                   q=_rotate(graph.q[layer], lengths - 1, 1e6))
        outs.append(_decode_exact(one, lengths))
    return {"out": outs, "kv": kv}
