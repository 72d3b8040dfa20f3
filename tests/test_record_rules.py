"""The rules on record counts (csrc/srx_record_rules.h), compiled for the host: the estimate that a draw's lists are
first formed for has the draw's own size in it, and the tables sized for a capacity hold the parts and split tiles
of every draw within it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <random>
#include <vector>
#include "srx_record_rules.h"
using namespace srx;
int main() {
  std::mt19937_64 rng(1);
  int bad = 0;
  auto below = [&](uint64_t n) { return rng() % n; };
  for (int it = 0; it < 20000; ++it) {
    const uint32_t cap = uint32_t(1) << (8 + below(24)), total = uint32_t(below(uint64_t(cap) + 1));
    const uint32_t prims = uint32_t(1 + below(it % 2 ? 100000 : 1u << 30));
    uint32_t np, nt, parts = 0, tiles = 0;
    vis_split_bounds(prims, cap, &np, &nt);
    const uint32_t busy = uint32_t(below((1u << 18) + 1)), part = vis_part(prims, total, busy, vis_tile_cost(4, true));
    if (vis_can_split(prims)) {
      for (uint64_t left = total; left;) {  // lists just above a multiple of the part, or of any length
        uint64_t n = it % 3 ? part + 1 + part * below(3) : 1 + below(left);
        n = n < left ? n : left;
        left -= n;
        if (n > part) parts += uint32_t((n + part - 1) / part), ++tiles;
        if (!(it % 3) && left < total / 64) break;
      }
    }
    if (parts > np || tiles > nt) ++bad, std::printf("cap %u total %u prims %u: %u parts of %u, %u tiles of %u\n", cap, total, prims, parts, np, tiles, nt);
  }
  // a mesh of small triangles, and its neighbours on either side of the rule
  if (vis_large(24000, 16384) || vis_part(16384, 24000, 1024, 88) != VIS_PART_SMALL - 1) ++bad;
  if (vis_large(4 * 16384 - 1, 16384) || !vis_large(4 * 16384, 16384)) ++bad;
  if (vis_part(2000, 330000, 1024, 88) != VIS_PART_LARGE - 1 || vis_part(1u << 22, 6400000, 0, 160) != 10239) ++bad;
  // a mesh keeps room for its own triangles after any number of small draws; deep draws are remembered
  if (record_estimate(20000, 522242, 8160) != 3 * 522242 + 8160 || record_estimate(0, 522242, 8160) != 3 * 522242 + 8160) ++bad;
  if (record_estimate(330000, 2000, 1024) != 412500 || record_estimate(0, 12, 64) != 65536) ++bad;
  if (record_estimate(0xFFFFFFF0u, 1, 1) != MAX_RECORDS || record_estimate(0, 0x55554000u, 1 << 18) != MAX_RECORDS) ++bad;
  // the steps are in order, and a list is in the step that holds it
  for (uint32_t k = 0; k < VIS_STEPS; ++k) {
    const uint32_t a = vis_step_size(k), last = k + 1 < VIS_STEPS ? vis_step_size(k + 1) - 1 : 0xFFFFFFFFu;
    if (last <= a || vis_step(a) != k || vis_step(last) != k || vis_step(a + (last - a) / 2) != k) ++bad;
  }
  for (int it = 0; it < 100000; ++it) {  // the tiles that a part size splits are those of its step and above
    const uint32_t part = vis_part(1 + uint32_t(below(1u << 30)), uint32_t(below(1ull << 32)), uint32_t(below(1u << 18)), 160);
    const uint32_t n = it % 2 ? part + uint32_t(below(3)) : VIS_PART_SMALL + uint32_t(below(0xFFFFF000u));
    if ((n > part) != (n >= VIS_PART_SMALL && vis_step(n) >= vis_step(part + 1))) ++bad;
  }
  // lists that keep the pass waiting are split, lists of a pass that is busy for longer are not
  if (vis_part(522242, 560000, 1008, vis_tile_cost(4, true)) > 1500 || vis_part(522242, 910000, 6500, vis_tile_cost(4, true)) < 2800) ++bad;
  if (vis_can_split(682) || !vis_can_split(683)) ++bad;
  return bad != 0;
}
"""


def test_rules_on_the_host(tmp_path):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "salviarenderer_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
