"""The size rules of zeknox_amd/csrc/tuning.h (host code, compiled here)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "zeknox_amd", "csrc")
DEFAULT, NEVER = 1 << 20, (1 << 64) - 1

PROGRAM = """
#include <stdio.h>
#include "tuning.h"
int main()
{
    unsigned long long n, h, least;
    while (scanf("%llu %llu %llu", &n, &h, &least) == 3)
        printf("%u %d %d\\n", zkx::lone_tree_tile_log(n, h, least), (int)zkx::lone_tree_levels_apart(n, h, least),
               (int)zkx::lone_tree_narrow(n, h, least));
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r")], check=True)

    def ask(*cases):
        out = subprocess.run([str(d / "r")], input="".join("%d %d %d\n" % c for c in cases), check=True, capture_output=True,
                             text=True).stdout.split("\n")
        return [tuple(map(int, line.split())) for line in out[:-1]]
    return ask


def test_lone_trees(rules):
    sizes = [1 << k for k in range(0, 33)]
    for ht, switch in ((0, 16), (3, 16), (1, 18), (4, 18), (2, 15)):
        small = ht in (0, 3)
        for lg, (tile, apart, narrow) in enumerate(rules(*[(n, ht, DEFAULT) for n in sizes])):
            assert apart == (lg >= switch) and narrow == (small and lg < switch)
            # 2^8: leaves alone, or a tree that does not fill the chip with larger tiles
            assert tile == ((8 if lg <= 16 else min(lg - 8, 10)) if ht == 2 else 9 if lg == 17 and not (apart or small) else 8)
        for lg, (tile, apart, narrow) in enumerate(rules(*[(n, ht, NEVER) for n in sizes])):
            assert not apart and narrow == (small and lg <= 15)
            assert tile == (8 if lg <= 16 else lg - 8 if lg <= 18 else 10 if ht == 2 else 9 if small else 8)
        for tile, apart, narrow in rules(*[(n, ht, 0) for n in sizes]):
            assert (apart, narrow) == (1, 0) and (tile == 8 or ht == 2)
