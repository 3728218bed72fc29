"""How prefill calls are cut (pda_prefill_plan.h, plain host code), built into a
small program and read on the CPU: the query blocks per wave on both sides of
each line of the rule, and over a sweep that the two-block kernel never gets
more of a CU's time than the one-block one, nor a window or softcap."""

import shutil
import subprocess
from pathlib import Path

import pytest

from instinct_amd import _lib

CSRC = Path(__file__).resolve().parent.parent / "llm-inference_amd" / "csrc"
CXX = shutil.which("g++") or shutil.which("clang++")

pytestmark = pytest.mark.skipif(CXX is None, reason="no C++ compiler")

PROGRAM = r"""
#include <stdio.h>
#include "pda_prefill_plan.h"
int main() {
  int start, count, heads, dim, window, request;
  float cap;
  while (scanf("%d %d %d %d %d %f %d", &start, &count, &heads, &dim, &window, &cap, &request) == 7) {
    using namespace pda_prefill;
    const int s = prefill_splits(start, count, heads, prefill_dim(dim), window, request);
    printf("%d %d %zu\n", s, query_blocks(start, count, heads, dim, window, cap, s),
           prefill_workspace(s, count, heads, prefill_dim(dim)));
  }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    out = tmp_path_factory.mktemp("plan")
    (out / "plan.cpp").write_text(PROGRAM)
    subprocess.run([CXX, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", "plan.cpp", "-o", "plan"],
                   cwd=out, check=True)

    def run(cases):
        text = "".join(" ".join(map(str, c)) + "\n" for c in cases)
        lines = subprocess.run([out / "plan"], input=text, capture_output=True, text=True,
                               check=True).stdout.splitlines()
        return [tuple(map(int, line.split())) for line in lines]

    return run


def test_query_blocks(plan):
    # start, count, q heads, head dim, window, softcap, requested ranges: blocks
    want = {
        (32256, 512, 28, 128, 0, 0, 0): 2,
        (7680, 512, 28, 128, 0, 0, 0): 2, (7679, 512, 28, 128, 0, 0, 0): 1,   # 8192 keys
        (32256, 512, 28, 64, 0, 0, 0): 1, (32256, 512, 28, 256, 0, 0, 0): 1,
        (32256, 512, 28, 96, 0, 0, 0): 1, (32256, 512, 28, 112, 0, 0, 0): 1,
        (32256, 512, 28, 128, 32768, 0, 0): 2,  # a window over every key
        (32256, 512, 28, 128, 32767, 0, 0): 1, (0, 8192, 28, 128, 1024, 0, 0): 1,
        (32256, 512, 28, 128, 0, 50, 0): 1,
        (32256, 1152, 28, 128, 0, 0, 0): 1,  # 280 workgroups of 256 in 2 ranges
        (32256, 640, 28, 128, 0, 0, 0): 2, (32256, 384, 28, 128, 0, 0, 0): 1,
        (32256, 3000, 28, 128, 0, 0, 0): 1, (8192, 4096, 28, 128, 0, 0, 0): 2,
        (8192, 256, 8, 128, 0, 0, 0): 1,     # ranges of 528 keys
        (32256, 512, 28, 128, 0, 0, 32): 2, (32256, 512, 28, 128, 0, 0, 36): 1,  # 910 keys
    }
    assert [p[1] for p in plan(want)] == list(want.values())


def test_the_gpu_tests_shapes_take_two_blocks(plan):
    from test_gpu_prefill_pipelined import TWO_BLOCKS

    cases = [(start, count, hq, 128, window, 0, splits)
             for hq, count, start, _, window, splits, _ in TWO_BLOCKS]
    assert [p[1] for p in plan(cases)] == [2] * len(cases)


def test_two_blocks_cost_no_more_of_a_cu(plan):
    cases = [(start, count, heads, 128, window, cap, request)
             for start in (0, 1, 7000, 8192, 32256, 100000)
             for count in (1, 100, 129, 256, 300, 512, 640, 1152, 2050, 4096, 8192, 20000)
             for heads in (1, 8, 14, 28, 32, 40, 64)
             for window in (0, 512, 8192, 1 << 20)
             for cap in (0, 50) for request in (0, 1, 7)]
    two = 0
    for case, (splits, blocks, _) in zip(cases, plan(cases), strict=True):
        start, count, heads, _, window, cap, _ = case
        assert blocks in (1, 2)
        if blocks == 2:
            two += 1
            groups = [-(-count // q) * heads * splits for q in (128, 256)]
            assert 2 * -(-groups[1] // 256) <= -(-groups[0] // 256), case
            assert not cap and (not window or window >= start + count), case
    assert two > 100


def test_workspace_of_the_plan(plan):
    """What pda_prefill_workspace_bytes reports is the plan of the call, of
    either cache type: bytes where there are ranges, none where there is one."""
    cases = [(start, count, heads, dim, window, 0, request)
             for start in (0, 500, 7040, 32256) for count in (1, 512, 1152, 4224)
             for heads in (8, 28, 32) for dim in (64, 80, 96, 128, 256, 512)
             for window in (0, 700) for request in (0, 3)]
    for case, (splits, _, nbytes) in zip(cases, plan(cases), strict=True):
        start, count, heads, dim, window, _, request = case
        assert _lib.prefill_workspace_bytes(start, count, heads, dim, window, request) == (
            splits, nbytes), case
        assert (splits > 1) == (nbytes > 0), case
    # 16-bit calls of this shape once planned one range and 8-bit ones two.
    assert _lib.prefill_workspace_bytes(32256, 1152, 28, 128) == (
        2, 2 * 1152 * 28 * 128 * 4 + 2 * 1152 * 28 * 8)
