"""How the groups of a crowded bucket are dealt to the parts that share it (csrc/bucket_deal.h, used by the transposing
SpMV without preprocess): every group to one part, and the work even over all wavefronts of all parts.  Needs no GPU."""
import subprocess

from mcsparse_amd import build

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "bucket_deal.h"
int main() {
    const uint32_t waves = 16;
    for (uint32_t parts = 2; parts <= 40; ++parts) {
        for (uint32_t groups = 1; groups <= 2100; groups += groups < 70 ? 1 : 61) {
            std::vector<uint32_t> taken(parts * waves, 0);
            for (uint32_t g = 0; g < groups; ++g) {
                const uint32_t part = mcsp::part_of_group(g, waves, parts);
                if (part >= parts) return std::printf("group %u of %u parts: %u\n", g, parts, part), 1;
                ++taken[part * waves + g % waves];
            }
            // a wavefront walks ceil(groups / waves) groups at most, and its parts take turns along the walk
            const uint32_t walk = (groups + waves - 1) / waves, most = (walk + parts - 1) / parts;
            const uint32_t busiest = *std::max_element(taken.begin(), taken.end());
            if (busiest > most) return std::printf("%u groups, %u parts: %u, not %u\n", groups, parts, busiest, most), 1;
            // and every part gets its share of the groups, one per wavefront more or less
            for (uint32_t p = 0; p < parts; ++p) {
                uint32_t sum = 0;
                for (uint32_t w = 0; w < waves; ++w) sum += taken[p * waves + w];
                if (sum > groups / parts + waves || sum + waves < groups / parts)
                    return std::printf("%u groups, %u parts: part %u has %u\n", groups, parts, p, sum), 1;
            }
        }
    }
    // sixteen groups, one to a wavefront: no part has more than its share
    for (uint32_t parts = 2; parts <= 16; ++parts) {
        std::vector<uint32_t> sum(parts, 0);
        for (uint32_t g = 0; g < waves; ++g) ++sum[mcsp::part_of_group(g, waves, parts)];
        if (*std::max_element(sum.begin(), sum.end()) > (waves + parts - 1) / parts) return std::printf("one round\n"), 1;
    }
    return std::puts("ok"), 0;
}
"""


def test_groups_are_dealt_evenly(tmp_path):
    src, exe = tmp_path / "deal.cpp", tmp_path / "deal"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", build.CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout
