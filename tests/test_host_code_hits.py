"""Which bits of the byte-code matches belong to elements of the row (dt_codes.h, compiled here): a row
fills whole words of four elements, word j of thread t holding elements 4 (1024 j + t) .. + 3, and a
thread's words start at a multiple of 16 of its 64."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "turbo-winfare_amd" / "csrc"
PROGRAM = """
#include <cstdio>
#include "dt_codes.h"
int main() {
    for (unsigned first = 0; first < 64; first += 8)
        for (unsigned words = 0; words <= 64; ++words) std::printf("%u\\n", tdt::filled_hits(first, words));
}
"""


def test_hits_past_the_row_are_dropped(tmp_path):
    (tmp_path / "hits.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", f"-I{CSRC}", str(tmp_path / "hits.cpp"), "-o", str(tmp_path / "hits")], check=True)
    got = iter(map(int, subprocess.run([str(tmp_path / "hits")], check=True, capture_output=True, text=True).stdout.split()))
    for first in range(0, 64, 8):
        for words in range(65):
            want = sum(1 << (8 * e + 7 - w) for w in range(8) for e in range(4) if first + w < words)
            assert next(got) == want, (first, words)
