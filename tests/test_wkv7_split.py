"""The rule that spreads the heads of the chunked WKV-7 scan over workgroups
(``csrc/wkv7_split.h``, host arithmetic), compiled with g++ and asked directly."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "yufmusicgen_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

MAIN = r"""
#include "wkv7_split.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char **argv) {
    for (int i = 1; i + 4 < argc; i += 5)
        std::printf("%d\n", yuf::wkv7_value_tiles(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]),
                                                  std::atoi(argv[i + 3]) != 0, argv[i + 4][0] == '-' ? nullptr : argv[i + 4]));
}
"""


@pytest.fixture(scope="module")
def value_tiles(tmp_path_factory):
    d = tmp_path_factory.mktemp("split")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(d / "split")],
                   check=True)

    def ask(nb, heads, call_heads=0, two=True, force="-"):
        out = subprocess.run([str(d / "split"), str(nb), str(heads), str(call_heads), str(int(two)), force],
                             capture_output=True, text=True, check=True)
        return int(out.stdout)

    return ask


@pytest.mark.parametrize("nb,heads,call,two,want", [
    (1, 16, 0, True, 0), (2, 128, 0, True, 1), (2, 129, 0, True, 0),
    (3, 85, 0, True, 1), (3, 86, 0, True, 2), (3, 128, 0, True, 2), (3, 129, 0, True, 0),
    (4, 64, 0, True, 1), (4, 65, 0, True, 2), (4, 128, 0, True, 2), (4, 129, 0, True, 0),
    (3, 16, 64, True, 1), (3, 24, 96, True, 2), (3, 32, 128, True, 2),   # parts of a prefill: all of them run at once
    (3, 80, 160, True, 0), (3, 128, 256, True, 0),
    (4, 64, 0, False, 1), (4, 65, 0, False, 0),                          # no pair form with the model's prep
    (4, 24, 96, False, 1), (4, 32, 128, False, 1), (4, 64, 129, False, 0), (4, 96, 192, False, 0),
])
def test_form_follows_the_heads_that_run_at_once(value_tiles, nb, heads, call, two, want):
    assert value_tiles(nb, heads, call, two) == want


@pytest.mark.parametrize("nb,heads,two,force,want", [
    (3, 16, True, "0", 0), (3, 1000, True, "1", 2), (3, 16, True, "1", 1), (3, 16, True, "2", 2), (3, 1000, True, "4", 1),
    (4, 16, False, "2", 0), (4, 1000, False, "1", 0), (4, 1000, False, "4", 1),
    (3, 1000, True, "on", 2), (3, 1000, True, "true", 2), (3, 16, True, "", 1), (3, 1000, True, "00", 2),
])
def test_forced_forms(value_tiles, nb, heads, two, force, want):
    assert value_tiles(nb, heads, 0, two, force) == want
