"""Offsets of the rows that a tile of cached keys reads (csrc/kernels/span_rows.h), against 64 bits: short caches and ones whose distances pass 32 bits as bytes."""
import os
import subprocess

import espresso_amd._lib as lib

SOURCE = r"""
#include <cstdio>
#include "kernels/span_rows.h"
int main() {
    const long long far[] = {0, 1, 30, 31, 32, 33, 63, 1000, 65535, 131072, 262143, 262144, 262149, 524287, 524288, 524293, 1048576, 1048580, 2097151, 2097157, 16777221};
    for (int heads = 1; heads <= 128; heads *= 2)
        for (int size = 64; size <= 128; size *= 2) {
            const unsigned row_bytes = heads * size * 2;
            for (long long distance : far)
                for (int row = 0; row < esp::kSpanTile; row++) {
                    const unsigned most = esp::last_row_offset((int)distance, row_bytes), own = row * row_bytes, at = own < most ? own : most;
                    if (at != (row < distance ? row : distance) * row_bytes) { std::printf("%d heads of %d, distance %lld, row %d: %u\n", heads, size, distance, row, at); return 1; }
                }
            if (esp::last_row_offset(-1, row_bytes) || esp::last_row_offset(-224, row_bytes)) { std::puts("a tile behind the last key"); return 1; }
        }
    return 0;
}
"""


def test_rows_of_a_tile_end_at_the_last_key_however_far_it_is(tmp_path):
    source, program = tmp_path / "rows.cpp", tmp_path / "rows"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(os.path.dirname(lib.__file__), "csrc"), str(source), "-o", str(program)], check=True)
    got = subprocess.run([str(program)], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout
