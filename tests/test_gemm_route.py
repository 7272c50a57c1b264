"""The kernel and the K split that dnx_gemm_q8 / _q4 choose by shape, from the
header that holds the rules (host code alone, compiled here)."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "dianoia_amd", "csrc")

MAIN = r"""
#include <stdio.h>
#include "gemm_route.h"
int main() {
  int q4;
  long long rows, cols, n;
  while (scanf("%d %lld %lld %lld", &q4, &rows, &cols, &n) == 4) {
    const dnx::GemmKernel k = dnx::gemm_kernel_for(q4 != 0, rows, cols, n);
    const char* names[] = {"skinny", "chunk1", "chunk2", "tile32", "tile64"};
    const bool t32 = k == dnx::GemmKernel::kTile32, t64 = k == dnx::GemmKernel::kTile64;
    int splits = 1;
    if (t32 || t64) {
      const int64_t tiles = t32 ? (rows + 127) / 128 : (rows + 63) / 64 * ((n + 63) / 64);
      const int stages = (int)((cols / 32 + dnx::kTileBlocks - 1) / dnx::kTileBlocks);
      const int per = dnx::tile_split_stages(tiles, stages);
      splits = (stages + per - 1) / per;
    }
    printf("%s %d\n", names[(int)k], splits);
  }
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", str(d / "main"),
                    str(d / "main.cpp")], check=True)

    def ask(shapes):
        text = "".join("%d %d %d %d\n" % s for s in shapes)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True,
                             check=True).stdout
        return [(a, int(b)) for a, b in (line.split() for line in out.splitlines())]

    return ask


def test_short_k_keeps_the_tile_kernel(route):
    """K <= 128 is one stage of the tile kernel, without a reduce: the chunk
    kernel takes it only where it measured faster (one token group, K <= 96)."""
    shapes = [(q4, rows, cols, n) for q4 in (0, 1) for cols in (32, 64, 96, 128)
              for rows, n in ((353, 64), (569, 460), (2941, 121), (4373, 56), (79, 373))]
    for (q4, rows, cols, n), (kernel, splits) in zip(shapes, route(shapes)):
        one_group = -(-rows // 32) * -(-n // 32) <= 256
        assert kernel == ("chunk1" if one_group and cols <= 96 else "tile64"), (rows, cols, n)
        assert splits == 1


def test_chunk_lines(route):
    """Either side of the other lines of the rule."""
    for shape, want in [((0, 3072, 1024, 16), "skinny"), ((0, 3072, 1024, 17), "chunk1"),
                        ((0, 3072, 1024, 64), "chunk1"), ((0, 3072, 1024, 128), "chunk2"),
                        ((0, 3072, 1024, 200), "tile64"), ((1, 2048, 2048, 64), "chunk1"),
                        ((1, 2048, 2048, 33), "tile64"), ((0, 512, 2048, 64), "tile64"),
                        ((0, 1024, 2080, 64), "tile64"), ((0, 512, 160, 17), "chunk1"),
                        ((1, 4096, 2080, 8), "tile32"), ((1, 4096, 2080, 17), "tile32")]:
        assert route([shape])[0][0] == want, shape


def test_calls_that_allocate_nothing(route):
    """dnx_kernels.h names the calls that take no memory of the library's own,
    so that a caller may capture them at once: none of them splits K, and the
    sentence names no more than that."""
    sizes = [1, 31, 32, 33, 512, 2048, 3072, 8192, 8193, 20000, 151936]
    shapes = [(q4, rows, cols, n) for q4 in (0, 1) for rows in sizes
              for cols in (32, 64, 128, 160, 512, 992, 1024, 1056, 2048, 2080, 4096)
              for n in (1, 5, 16, 17, 32, 33, 63, 64, 65, 128, 200, 512, 1024)]
    named = 0
    for (q4, rows, cols, n), (kernel, splits) in zip(shapes, route(shapes)):
        if (n <= 16 and cols <= 2048) or (cols <= 1024 and -(-rows // 32) * -(-n // 64) <= 256):
            named += 1
            assert splits == 1, (q4, rows, cols, n, kernel)
    assert named > 800
    header = open(os.path.join(CSRC, "..", "..", "include", "dnx_kernels.h")).read()
    header = " ".join(header.replace("//", " ").split())
    assert ("n <= 16 with K <= 2048, and K <= 1024 where ceil(rows / 32) * ceil(n / 64) <= 256. "
            "Any other call may split K") in header
    # Two that a line at K <= 2048 alone would name: they split K.
    for shape in ((0, 512, 2048, 64), (1, 2048, 2048, 33)):
        assert route([shape])[0][1] > 1
