"""The levels of the build's table of unions, at every size where their number changes and up to the largest scene."""
import subprocess

from raytracergpu_mastersproject_amd import build as B

SRC = r"""
#include <cstdio>
#include <vector>
#include "box_levels.hpp"
using namespace rtgpu;
int main() {
    std::vector<uint32_t> sizes = {(1u << 27) - 17u};
    for (uint32_t k = 0; k < 27; ++k)
        for (int d = -2; d <= 2; ++d)
            if ((int64_t)(1u << k) + d > 0) sizes.push_back((1u << k) + d);
    for (uint32_t n : sizes) {
        uint64_t written = 0, levels = 0;
        for (uint32_t level = 0; box_count(n, level) > 1u; level += 8) {  // one launch: levels level + 1 .. level + 8
            uint64_t at = boxes_before(n, level + 1u);
            for (uint32_t k = 1; k <= 8u; ++k) {
                const uint64_t count = box_count(n, level + k);
                if (count != ((uint64_t)n >> (level + k)) || at != written || at + count > n) {
                    std::printf("n %u level %u: %llu boxes at %llu\n", n, level + k, (unsigned long long)count, (unsigned long long)at);
                    return 1;
                }
                at += count;
                written += count;
                levels += count > 0;
            }
        }
        if (n > 1 && (n >> levels) != 1u) { std::printf("n %u: %llu levels\n", n, (unsigned long long)levels); return 1; }
    }
    return 0;
}
"""


def test_levels_follow_one_another(tmp_path):
    (tmp_path / "levels.cpp").write_text(SRC)
    exe = tmp_path / "levels"
    subprocess.run(["g++", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", f"-I{B.CSRC}",
                    str(tmp_path / "levels.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
