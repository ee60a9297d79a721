"""CPU-only checks of rules that choose a launch's shape: small programs over the kernels' own headers, linked with the built library where the rule
lives in it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qingming-qwen3-tts_amd", "csrc")
LIB = os.path.join(ROOT, "qingming-qwen3-tts_amd", "lib")


def run(tmp_path, source, library=None):
    """The output lines of a program of one `main`."""
    path = tmp_path / "rule.cpp"
    path.write_text(source)
    link = ["-L" + LIB, "-l" + library, "-Wl,-rpath," + LIB] if library else []
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), "-o",
                    str(tmp_path / "rule"), str(path), *link], check=True)
    return subprocess.run([str(tmp_path / "rule")], check=True, capture_output=True, text=True).stdout.splitlines()


def test_a_rounded_grid_keeps_no_die_longer_than_an_even_deal(tmp_path):
    """Row linears: blocks go to the eight dies of 32 CUs in turn, one to a CU.  Whatever the grid's width is rounded to, no die walks more rounds of
    blocks than all of them do when the tiles are dealt out one by one; and where that holds, many column tiles are rounded."""
    lines = run(tmp_path, """
#include <cstdio>
#include "qm_linear_rows_params.h"
int main() {
    for (int columns = 1; columns <= 400; ++columns)
        for (int rows = 1; rows <= 64; ++rows)
            for (int pieces = 1; pieces <= 8; pieces *= 2) std::printf("%d %d %d %d\\n", columns, rows, pieces, qm::rows_grid_columns(columns, rows, pieces));
}""")
    assert len(lines) == 400 * 64 * 4
    rounded = 0
    for line in lines:
        columns, rows, pieces, width = map(int, line.split())
        assert width in (columns, (columns + 7) // 8 * 8)
        tiles = columns * rows * pieces
        if width % 8 == 0:                                   # column c's tiles are all on die c % 8
            busiest = -(-columns // 8) * rows * pieces
        else:                                                # the grid has a tile for every block: dealt out one by one
            assert width == columns
            busiest = -(-tiles // 8)
        if width != columns:
            assert -(-busiest // 32) <= -(-(-(-tiles // 8)) // 32), line
            rounded += 1
    assert rounded > 5000
    assert "81 8 1 88" in lines and "42 6 1 42" in lines and "42 3 2 42" in lines
