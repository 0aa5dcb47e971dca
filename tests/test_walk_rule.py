"""The rule that walks the rows of a tree on every row through it at its end, in a host program (no GPU)."""
import os
import subprocess

RULE = r"""
#include "walk_rule.h"
#include <cstdio>
int main() {
    struct { int64_t rows; int all_feats, feats, depth; bool oblivious, walk; } t[] = { // the faster of the two, by 1 to 162 us a round
        {1000000, 100, 100, 11, false, true}, {4000000, 20, 20, 11, false, true}, {10000000, 100, 100, 6, false, true}, {10000000, 100, 100, 8, false, true},
        {10000000, 100, 100, 11, false, false}, {4000000, 100, 100, 11, false, false}, {10000000, 20, 20, 11, false, true}, {10000000, 50, 50, 11, false, true},
        {10000000, 100, 50, 11, false, true}, // half the columns sampled: at most 50 bytes a row
        {10000000, 100, 100, 9, true, true}, {10000000, 100, 100, 11, true, true}, {4000000, 100, 100, 8, true, true}, {4000000, 100, 100, 11, true, true}};
    for (const auto &c : t)
        if (walk_pays(c.rows, c.all_feats, c.feats, c.depth, c.oblivious) != c.walk) return printf("%lld x %d depth %d\n", (long long)c.rows, c.feats, c.depth), 1;
    for (int depth = 1; depth <= 40; depth++) // an oblivious tree tests a feature a level: never the more bytes
        for (int feats = 1; feats <= 4000; feats = feats * 3 + 1)
            if (!walk_pays(100000000, 4000, feats, depth, true)) return printf("depth %d, %d features\n", depth, feats), 2;
}
"""


def test_rows_are_walked_where_it_was_faster(evt, tmp_path):
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.cpp").write_text(RULE)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-x", "c++", "-O0", "-std=c++17", "-I", csrc, str(tmp_path / "main.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
