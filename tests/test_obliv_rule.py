"""The rule that takes an oblivious level to the one-launch kernel against the list of that kernel's instances, in a host program (no GPU)."""
import os
import subprocess

RULE = r"""
#include "obliv_rule.h"
#include <cstdio>
#include <initializer_list>
int main() { // every channel count, bin count and level: accepted within the words' budget, and each then has one instance and fits its arrays
    int accepted = 0;
    for (int channels : {2, 3, 5})
        for (int bins = 2; bins <= 255; bins++)
            for (int nodes = 1; nodes <= 1 << 15; nodes *= 2) {
                const bool want = bins >= 4 && nodes <= 32 && nodes * channels * ((bins + 63) / 64) <= 192;
                if (obliv_level_fits(channels, bins, nodes) != want) return printf("%d channels %d bins %d nodes\n", channels, bins, nodes), 1;
                if (!want) continue;
                int found = 0;
#define ONE(C_, L_, W_) found += channels == C_ && obliv_lane_bins(bins) == L_ && obliv_wave_nodes(nodes) == W_;
                EVT_OBLIV_LEVELS(ONE)
                const int threads = 64 * (nodes < 4 ? 4 : nodes > 16 ? 16 : nodes), most = channels * obliv_lane_bins(bins) > 12 ? 512 : 1024;
                if (found != 1 || 64 * obliv_lane_bins(bins) < bins || threads / 64 * obliv_wave_nodes(nodes) < nodes || threads < 3 * nodes ||
                    threads < channels * nodes || threads > most || nodes * bins * 8 + 2 * 32 * channels * 8 + 64 > 65536 || channels > 2 * bins)
                    return printf("%d channels %d bins %d nodes: %d\n", channels, bins, nodes, found), 2;
                accepted++;
            }
    printf("%d\n", accepted);
}
"""


def test_every_level_the_rule_takes_has_its_kernel(evt, tmp_path):
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.cpp").write_text(RULE)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-x", "c++", "-O0", "-std=c++17", "-I", csrc, str(tmp_path / "main.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
    assert int(run.stdout) > 3000  # levels
