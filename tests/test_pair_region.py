"""The digest's region arithmetic (csrc/pair_region.hpp) walked on the host as
the kernel walks it: every start below, at and past the end of an even and an
odd buffer, every count, every lane's loads; none may lie outside the buffer,
and each pair of the region that the buffer holds is added once."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gat_amd" / "csrc"

WALK = r"""
#include <cstdio>
#include <vector>
#include "pair_region.hpp"
using namespace gat;
int main() {
  constexpr uint64_t kSpan = 16;  // pairs a workgroup takes at a time, two per lane
  const uint64_t far[] = {uint64_t(1) << 33, (uint64_t(1) << 33) + 1, ~uint64_t(0) - 1, ~uint64_t(0)};
  for (uint64_t cap = 0; cap <= 37; ++cap)
    for (uint64_t k = 0; k < 84; ++k)
      for (uint64_t count = 0; count <= 48; ++count)
        for (uint64_t split = 1; split <= 3; ++split) {
          const uint64_t base = k < 80 ? k : far[k - 80];
          const PairRegion r = pair_region(base, count, cap);
          std::vector<int> added(cap);
          for (uint64_t y = 0; y < split; ++y) {
            if (r.first + y * kSpan >= r.end) continue;
            for (uint64_t s = r.first + y * kSpan; s < r.end; s += split * kSpan)
              for (uint64_t at = s; at < s + kSpan; at += 2) {
                if (whole_groups(r.end, cap)) {  // load_pair2_in reads two pairs
                  const uint64_t g = clamped_group(at, r.end);
                  if (g + 1 >= cap) return std::printf("group %llu of %llu\n", (unsigned long long)g, (unsigned long long)cap), 1;
                } else if (at + 1 < r.end) {     // load_pair2: two
                  if (at + 1 >= cap) return std::printf("pair %llu of %llu\n", (unsigned long long)at + 1, (unsigned long long)cap), 1;
                } else if (at < r.end && at >= cap) {  // or the lone last one
                  return std::printf("lone pair %llu of %llu\n", (unsigned long long)at, (unsigned long long)cap), 1;
                }
                if (at >= r.begin && at < r.end) ++added[at];
                if (at + 1 < r.end) ++added[at + 1];
              }
          }
          for (uint64_t i = 0; i < cap; ++i)
            if (added[i] != (i >= base && i - base < count ? 1 : 0))
              return std::printf("pair %llu added %d times\n", (unsigned long long)i, added[i]), 1;
        }
  return 0;
}
"""


def test_digest_loads_stay_inside_the_buffer(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
