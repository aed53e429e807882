"""The rule that chooses a prefill product's tiles (``csrc/gemm_tiles.h``, host
arithmetic), compiled with g++ and asked at shapes where one kernel is clearly
the faster one on an MI355X."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "yufmusicgen_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

MAIN = r"""
#include "gemm_tiles.h"
#include <cstdio>
#include <cstdlib>
int main(int, char **a) {
    const int n = std::atoi(a[1]), rows = std::atoi(a[2]), N = std::atoi(a[3]);
    yuf::TileProduct p[6];
    for (int i = 0; i < n; ++i) p[i] = {rows, N};
    const yuf::TileCost *t = yuf::ps_tile_rule(p, n, std::atoi(a[4]), std::atoi(a[5]), std::atoi(a[6]), false);
    std::printf("%d %d\n", t ? t->bm : 0, t ? t->bn : 0);
}
"""
MODES = {"planes": 0, "f32": 1, "bf16": 2, "small": 3}


@pytest.fixture(scope="module")
def tile(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(d / "tiles")],
                   check=True)

    def ask(form, rows, cols, depth, products=1):
        big = 0 if form == "small" else next(w for w in (256, 160, 128, 64) if cols % w == 0)
        out = subprocess.run([str(d / "tiles"), *map(str, (products, rows, cols, depth, MODES[form], big))],
                             capture_output=True, text=True, check=True)
        return tuple(int(x) for x in out.stdout.split())

    return ask


@pytest.mark.parametrize("form,rows,cols,depth,products,want", [
    # Large tiles: slower on small ones by 2-22 %.
    ("f32", 1300, 8192, 1024, 1, (0, 0)), ("f32", 2048, 5120, 640, 1, (0, 0)), ("f32", 12000, 1024, 4096, 1, (0, 0)),
    ("f32", 6500, 8192, 1024, 1, (0, 0)), ("planes", 5000, 20480, 640, 1, (0, 0)), ("planes", 5000, 5120, 640, 1, (0, 0)),
    ("planes", 16384, 5120, 640, 1, (0, 0)), ("planes", 16384, 64, 640, 3, (0, 0)), ("planes", 4096, 640, 128, 1, (0, 0)),
    ("planes", 8192, 192, 640, 1, (0, 0)), ("planes", 4000, 448, 640, 1, (0, 0)), ("planes", 8192, 576, 640, 1, (0, 0)), ("planes", 2048, 576, 640, 1, (0, 0)),
    ("bf16", 16384, 1024, 4096, 1, (0, 0)),
    # Small tiles: faster on them by 5 % to seven times.
    ("planes", 333, 640, 2560, 1, (32, 32)), ("planes", 1000, 5120, 640, 1, (64, 64)), ("planes", 4000, 5120, 640, 1, (128, 128)),
    ("planes", 2048, 64, 640, 1, (32, 32)), ("f32", 4000, 5120, 640, 1, (128, 128)), ("f32", 1000, 1024, 1024, 1, (64, 64)),
    ("bf16", 2200, 1024, 4096, 1, (64, 64)), ("bf16", 1700, 5120, 640, 1, (64, 128)), ("small", 100, 640, 640, 1, (32, 32)),
])
def test_tiles(tile, form, rows, cols, depth, products, want):
    assert tile(form, rows, cols, depth, products) == want
