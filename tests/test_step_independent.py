"""Whether a step's appends may run together (DecodeStepGraph._independent), on
CPU tensors: buffers of their own, shared arenas, views that overlap, layers of
different forms. An eager step asks before every run, so layers over shared
arenas must be told from the arenas alone."""

import pytest
import torch

from instinct_amd.step import DecodeStepGraph


def step(layers=3, heads=2, scales=False):
    s = DecodeStepGraph.__new__(DecodeStepGraph)
    half = lambda *shape: torch.zeros(shape, dtype=torch.float16)  # noqa: E731
    shapes = [(4, heads, 16, 64)] * 2 + [(4, heads, 16)] * 2 * scales
    s.arenas = [tuple(half(*shape) for shape in shapes) for _ in range(layers)]
    for name, n in (("q", 6), ("k", heads), ("v", heads), ("q_rot", 6), ("out", 6)):
        setattr(s, name, [half(5, n, 64) for _ in range(layers)])
    for name in ("slots", "positions", "tables", "lengths", "rows", "seq_tables", "workspace"):
        setattr(s, name, torch.zeros(8, dtype=torch.int32))
    return s


@pytest.mark.parametrize("layers,scales", [(1, False), (3, False), (3, True)])
def test_buffers_of_their_own(layers, scales):
    assert step(layers, scales=scales)._independent()


def test_shared_arenas_are_told_from_the_arenas():
    s = step(4)
    s.arenas = [s.arenas[i % 2] for i in range(4)]
    s.q = s.k = s.out = s.workspace = None  # not looked at
    assert not s._independent()


def test_overlaps():
    s = step()
    s.q[1] = s.out[0]
    assert not s._independent()
    s = step()
    s.k[2] = s.k[0].flatten()[64:].view(-1, 64)[:2]  # inside another layer's
    s.k[2] = s.k[2].view(1, 2, 64)
    assert not s._independent()
    s = step()
    s.arenas[1] = (s.arenas[1][0], s.arenas[0][1])  # values shared, keys not
    assert not s._independent()
    s = step()
    both = torch.zeros(2, 5, 6, 64, dtype=torch.float16)
    s.q[0], s.q[1] = both[0], both[1]  # neighbours
    assert s._independent()


def test_forms():
    s = step()
    s.arenas[2] = tuple(t.bfloat16() for t in s.arenas[2])
    assert not s._independent()
    s = step()
    s.arenas[2] += (torch.zeros(4, 2, 16), torch.zeros(4, 2, 16))
    assert not s._independent()
    s = step()
    s.q[2] = torch.zeros(5, 4, 64, dtype=torch.float16)
    assert not s._independent()


def test_empty_buffers():
    s = step()
    s.workspace = torch.zeros(0, dtype=torch.uint8)
    assert s._independent()
