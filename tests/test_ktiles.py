"""Positions along k of a tile product's loaders, on the host: ranges that one workgroup walks through for most of a
minute on the device."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "open-instruct_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "oi_ktiles.h"
int main(int argc, char** argv) {
    const int64_t ktiles = atoll(argv[1]), k_valid = atoll(argv[2]), bytes = 1024;
    KTiles<64> k((int)ktiles, k_valid);
    int64_t at = 0;
    for (int64_t t = 0; t < ktiles + 3; ++t) {
        const int64_t want = t < ktiles ? t : ktiles - 1;  // past the last k-tile: stays there
        const int64_t rows = k_valid - want * 64;
        const int64_t end = rows >= 64 ? 63 : rows - 1;
        if (at != want * bytes || (k.live != 0) != (t < ktiles)) { printf("k-tile %lld: at %lld\n", (long long)t, (long long)at); return 1; }
        if (t < ktiles && k.end_row() != end) { printf("k-tile %lld: last row %d\n", (long long)t, k.end_row()); return 1; }
        // a loader asks for its rows at the first k-tile and wherever this says so
        if (t > 0 && t < ktiles && end < 63 && !k.ending()) { printf("k-tile %lld: rows not asked for\n", (long long)t); return 1; }
        if (t >= ktiles && !k.ending()) { printf("past the end at %lld\n", (long long)t); return 1; }
        k.next();
        at += k.step(bytes);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    folder = tmp_path_factory.mktemp("ktiles")
    source, program = folder / "walk.cpp", folder / "walk"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(source), "-o", str(program)], check=True)
    return str(program)


# whole and ragged last k-tiles; rows that go on behind the range (a piece of a product cut along k); past 2^31 rows
@pytest.mark.parametrize(
    "ktiles,k_valid",
    [(1, 64), (1, 1), (2, 65), (3, 3 * 64 - 5), (5, 512), ((1 << 25) + 2, (1 << 31) + 128), ((1 << 25) + 2, (1 << 31) + 67)],
)
def test_every_k_tile_is_where_it_belongs(walk, ktiles, k_valid):
    res = subprocess.run([walk, str(ktiles), str(k_valid)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
