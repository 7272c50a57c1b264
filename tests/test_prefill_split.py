"""The prefill attention's split of its keys, from the header that holds the
rule (host code alone, compiled here)."""

import math
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "dianoia_amd", "csrc")

MAIN = r"""
#include <stdio.h>
#include "prefill_split.h"
int main() {
  long long position, n, heads, kv_heads, hd, window;
  while (scanf("%lld %lld %lld %lld %lld %lld", &position, &n, &heads, &kv_heads, &hd, &window) ==
         6) {
    const long long group = heads / kv_heads;
    const int gw = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const dnx::PrefillSplit s = dnx::prefill_split(position, n, heads, hd, window, gw);
    printf("%d %d %d %d %zu\n", s.splits, s.tps, s.kt, (int)s.panel, dnx::kPrefillWorkspace);
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("split")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", str(d / "main"),
                    str(d / "main.cpp")], check=True)

    def run(shapes):
        text = "".join(" ".join(map(str, s)) + "\n" for s in shapes)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True,
                             check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def test_no_later_call_allocates(ask):
    """Whatever call splits its keys first, its reserve holds for every other:
    positions, token counts, windows, head counts."""
    rng = random.Random(3)
    size = lambda low, high: int(math.exp(rng.uniform(math.log(low), math.log(high))))
    shapes = []
    for _ in range(20000):
        kv = rng.choice([1, 2, 3, 4, 5, 8, 16, 32])
        shapes.append((size(1, 40000) - 1, size(8, 3000), kv * rng.choice([1, 2, 3, 4, 6, 8, 16]),
                       kv, rng.choice([64, 128]), rng.choice([0, 0, size(1, 8192)])))
    split = 0
    for (position, n, heads, kv, hd, window), (splits, tps, kt, panel, reserve) in zip(
            shapes, ask(shapes)):
        split += splits > 1
        assert 1 <= splits <= 64 and (splits > 1 or not panel)
        if splits > 1:
            assert n * heads * splits * (hd + 4) * 4 <= reserve, (position, n, heads, kv, hd, window)
        # The splits hold the longest range of a workgroup's queries.
        group = heads // kv
        q = 64 // (4 if group % 4 == 0 else 2 if group % 2 == 0 else 1)
        longest = max(min(position + min(t + q, n), window + min(t + q, n) - t - 1 if window else
                          1 << 40) for t in range(0, n, q))
        assert splits * tps * kt >= longest > (splits - 1) * tps * kt
    assert split > 4000


def test_lines(ask):
    """Either side of the rule's lines: tiles of 32 keys at hd 64, one tile a
    split up to 9 MB of partials."""
    for shape, want in [((0, 32, 16, 4, 64, 0), (1, 1, 32)), ((0, 33, 16, 4, 64, 0), (1, 1, 64)),
                        ((0, 64, 16, 4, 64, 0), (1, 1, 64)), ((0, 65, 16, 4, 64, 0), (1, 3, 32)),
                        ((0, 96, 16, 4, 64, 0), (1, 3, 32)), ((0, 97, 16, 4, 64, 0), (2, 1, 64)),
                        ((256, 64, 16, 8, 128, 0), (10, 1, 32)),
                        ((269, 89, 32, 4, 128, 0), (6, 2, 32)),
                        ((2000, 8, 16, 8, 128, 0), (63, 1, 32)),
                        ((4095, 8, 16, 8, 128, 0), (43, 3, 32))]:
        assert ask([shape])[0][:3] == want, (shape, ask([shape])[0])
