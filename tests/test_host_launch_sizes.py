"""Launch sizes of the table repack over the whole range of accepted shapes (rows up to 2^24, in_dim
up to 8192), from the library's own host code compiled here: HIP refuses 2^32 threads or more in one
dimension of a grid, and both tables of a matrix share one launch."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "turbo-winfare_amd" / "csrc"
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "dt_grid.h"
int main(int argc, char** argv) {
    for (int i = 1; i < argc; ++i) std::printf("%u\\n", tdt::part_blocks(std::strtoull(argv[i], nullptr, 10), 256u));
}
"""
SHAPES = [(1, 64), (64, 64), (704, 2816), (262144, 2816), (1 << 24, 64), (1 << 24, 2816), (1 << 24, 5504),
          (1 << 24, 5824), (1 << 24, 8128), (1 << 24, 8192)]


@pytest.fixture(scope="module")
def part_blocks(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", f"-I{CSRC}", str(d / "grid.cpp"), "-o", str(d / "grid")], check=True)
    return lambda items: [int(v) for v in subprocess.run([str(d / "grid"), *map(str, items)], check=True,
                                                         capture_output=True, text=True).stdout.split()]


def test_both_tables_of_every_accepted_shape_fit_one_launch(part_blocks):
    for rows, in_dim in SHAPES:
        padded = (rows + 63) // 64 * 64
        weights, scales = padded * (in_dim // 32), padded * (in_dim // 64)
        w, s = part_blocks([weights, scales])
        assert 1 <= w and 1 <= s and (w + s) * 256 < 2**32, (rows, in_dim, w, s)
        for blocks, items in ((w, weights), (s, scales)):
            # one item to a thread until the cap, then whole turns of it
            assert blocks * 256 >= items or blocks * 256 == 2**30, (rows, in_dim, blocks)
            assert (blocks - 1) * 256 < items
