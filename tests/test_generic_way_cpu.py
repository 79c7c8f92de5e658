"""How chunk states of the sizes and types off the bf16 tilings are launched (csrc/ssd_cost.h: generic_way), against measured times.
The header is plain C++: compiled here with a small program around it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# type, headdim, dstate, chunk, 64 x 64 tiles per compute unit; microseconds with fp32 matrix instructions, with bf16 parts and a wave
# per tile, with parts and a quarter of a chunk per wave (8 or 24 heads, one group, inputs from memory)
MEASURED = [
    ('bf16', 32, 64, 100, 39.94, 53.7, 44.6, 66.0), ('bf16', 48, 32, 48, 39.94, 32.4, 38.0, 83.8),
    ('bf16', 48, 32, 128, 6.0, 14.5, 16.0, 16.7), ('bf16', 64, 64, 32, 6.0, 12.3, 10.3, 20.4),
    ('bf16', 128, 128, 32, 39.75, 51.9, 43.6, 115.3), ('bf16', 128, 128, 48, 6.0, 14.6, 12.0, 20.4),
    ('bf16', 128, 128, 100, 6.0, 23.8, 16.9, 21.4), ('fp16', 32, 32, 256, 6.0, 16.0, 18.1, 17.2),
    ('fp16', 32, 48, 48, 6.0, 9.1, 10.2, 14.0), ('fp16', 32, 64, 72, 0.5, 4.7, 8.1, 5.1),
    ('fp16', 32, 64, 160, 0.5, 5.2, 10.5, 6.0), ('fp16', 32, 64, 160, 24.0, 49.7, 37.6, 64.7),
    ('fp16', 48, 48, 48, 39.94, 45.7, 54.6, 110.9), ('fp16', 48, 48, 100, 1.0, 6.7, 11.1, 7.2),
    ('fp16', 48, 48, 160, 3.0, 13.3, 15.7, 16.2), ('fp16', 48, 64, 128, 6.0, 22.4, 18.8, 21.5),
    ('fp16', 48, 64, 128, 7.97, 27.4, 19.1, 26.4), ('fp16', 48, 64, 160, 7.97, 34.4, 21.7, 34.1),
    ('fp16', 48, 64, 256, 39.94, 170.9, 131.1, 160.3), ('fp16', 64, 32, 72, 2.0, 7.0, 9.4, 7.5),
    ('fp16', 64, 32, 128, 7.97, 21.3, 16.6, 21.6), ('fp16', 64, 32, 128, 12.0, 29.2, 21.4, 30.2),
    ('fp16', 64, 48, 72, 7.97, 30.0, 17.3, 31.9), ('fp16', 64, 48, 100, 7.97, 30.3, 20.1, 32.0),
    ('fp16', 64, 48, 256, 24.0, 109.6, 85.8, 111.8), ('fp16', 64, 64, 64, 7.97, 18.6, 14.8, 31.0),
    ('fp16', 64, 64, 64, 24.0, 47.3, 39.7, 83.9), ('fp16', 64, 64, 72, 24.0, 54.9, 45.6, 84.6),
    ('fp16', 64, 64, 128, 12.0, 47.1, 30.8, 45.6), ('fp16', 64, 64, 256, 7.97, 51.8, 32.6, 40.7),
    ('fp16', 64, 128, 72, 24.0, 54.2, 45.4, 83.2), ('fp16', 64, 128, 128, 8.06, 34.7, 28.3, 33.9),
    ('fp16', 64, 128, 128, 12.0, 46.2, 30.0, 45.0), ('fp16', 80, 80, 72, 2.0, 7.3, 9.9, 8.6),
    ('fp16', 80, 80, 72, 7.88, 18.5, 15.0, 24.2), ('fp16', 80, 80, 128, 12.0, 32.0, 24.0, 35.8),
    ('fp16', 80, 80, 160, 24.0, 62.7, 50.8, 86.5), ('fp16', 128, 128, 128, 39.75, 115.3, 84.0, 134.8),
    ('fp32', 32, 32, 32, 6.0, 7.3, 7.9, 13.0), ('fp32', 32, 32, 48, 6.0, 8.5, 9.6, 13.4),
    ('fp32', 32, 32, 100, 6.0, 11.2, 13.3, 14.4), ('fp32', 32, 32, 100, 39.94, 42.0, 49.7, 66.9),
    ('fp32', 32, 32, 128, 6.0, 11.8, 13.4, 14.9), ('fp32', 32, 48, 100, 39.94, 49.0, 57.2, 83.4),
    ('fp32', 32, 64, 100, 39.94, 59.0, 63.2, 91.4), ('fp32', 48, 32, 32, 39.94, 26.0, 33.5, 79.4),
    ('fp32', 48, 32, 100, 6.0, 13.3, 15.8, 17.6), ('fp32', 48, 48, 32, 6.0, 9.9, 10.6, 20.5),
    ('fp32', 48, 64, 72, 0.5, 5.2, 9.6, 5.9), ('fp32', 48, 64, 100, 3.0, 12.8, 13.7, 15.3),
    ('fp32', 48, 64, 128, 12.0, 40.5, 30.0, 48.1), ('fp32', 48, 64, 160, 2.0, 12.3, 15.2, 13.1),
    ('fp32', 64, 48, 32, 39.94, 45.7, 50.6, 124.3), ('fp32', 64, 128, 72, 0.5, 5.6, 10.7, 6.2),
    ('fp32', 64, 128, 100, 12.0, 44.6, 32.4, 47.1), ('fp32', 64, 128, 128, 3.94, 19.4, 16.1, 18.8),
    ('fp32', 80, 80, 48, 6.0, 10.5, 11.2, 19.5), ('fp32', 80, 80, 72, 2.0, 6.9, 9.2, 7.6),
    ('fp32', 80, 80, 100, 0.5, 5.6, 10.0, 6.1), ('fp32', 80, 80, 256, 4.12, 20.8, 23.3, 23.0),
]

PROGRAM = r"""
#include <cstdio>
#include "ssd_cost.h"
static int per_lane(int size) { const int tiles = (size + 63) / 64; return (size + 16 * tiles - 1) / (16 * tiles); }
int main()
{
    int P, N, Q, two; double tiles;
    while (std::scanf("%d %d %d %d %lf", &P, &N, &Q, &two, &tiles) == 5) {
        const ssd::cost::GenericWay w = ssd::cost::generic_way(Q, per_lane(P), per_lane(N), two != 0, N, tiles);
        std::printf("%d %d\n", (int)w.quarters, (int)w.parts);
    }
}
"""


@pytest.fixture(scope="module")
def way(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    assert cxx, "a C++ compiler is what builds the library"
    d = tmp_path_factory.mktemp("way")
    (d / "way.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-I", os.path.join(ROOT, "mamba-fused-minimal_amd", "csrc"), str(d / "way.cpp"), "-o", str(d / "way")], check=True)

    def ask(rows):
        text = "".join(f"{P} {N} {Q} {int(t != 'fp32')} {tiles}\n" for t, P, N, Q, tiles in rows)
        out = subprocess.run([str(d / "way")], input=text, stdout=subprocess.PIPE, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]
    return ask


def test_parts_are_taken_where_they_are_ahead(way):
    taken = 0
    for row, (quarters, parts) in zip(MEASURED, way([r[:5] for r in MEASURED])):
        former, wave, quarter = row[5:]
        if parts:
            taken += 1
            assert (quarter if quarters else wave) <= 1.04 * former, row
    assert taken >= 15


def test_without_parts_the_fp32_instructions_go_as_they_did(way):
    # one wave a tile in chunks up to 64 and from 24 tiles on, quarters elsewhere
    assert way([("fp32", 40, 40, Q, t) for Q, t in ((32, 1), (64, 30), (65, 1), (100, 23.9), (100, 24))]) == [(0, 0), (0, 0), (1, 0), (0, 1), (0, 0)]
    assert way([("fp16", 16, 128, Q, t) for Q, t in ((64, 3), (128, 12), (256, 30))]) == [(0, 0), (1, 0), (0, 0)]      # one row block


def test_sizes_that_are_tested_with_parts_run_them(way):
    # headdim, dstate, chunk and 64 x 64 tiles over 256 compute units of tests/test_gpu_split_products.py -> (quarters, parts)
    fp32 = [(64, 128, 257, 70 * 3 * 2), (64, 128, 257, 33 * 2 * 2), (63, 127, 257, 2 * 2 * 2), (64, 128, 100, 80 * 7 * 2), (48, 63, 100, 90 * 13), (48, 40, 100, 90 * 23)]
    two = [(64, 64, 257, 90 * 3), (31, 63, 257, 2 * 2), (64, 63, 64, 100 * 11), (32, 63, 100, 90 * 23), (64, 63, 100, 110 * 7)]
    assert way([("fp32", P, N, Q, t / 256) for P, N, Q, t in fp32]) == [(1, 1), (1, 1), (1, 1), (0, 1), (0, 1), (0, 1)]
    assert way([("fp16", P, N, Q, t / 256) for P, N, Q, t in two]) == [(1, 1), (1, 1), (0, 1), (0, 1), (0, 1)]
