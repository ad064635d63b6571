// Workgroup -> work-item maps of the prefill and backward grids, and the host-side
// choice of map for a launch. Plain integer C++: the functions are constexpr, so the
// kernels call them on the device (clang compiles constexpr functions for host and
// device) and tests/hip/grid_check.cpp, built by g++, checks on the CPU that every map
// the launchers select is a bijection from workgroup ids onto (unit, tile) pairs.
//
// The hardware deals linear workgroup ids round-robin to the 8 XCDs of MI355X
// (id % 8 = XCD); each XCD has its own L2, so the maps keep a unit's tiles (one
// (batch, head): the K/V, or Q/dO, they share) on one XCD.
#pragma once

#include <stdint.h>

namespace ffa {

// Launches of 257 to 512 workgroups, two to a CU, are resident all at once: the second 256
// join the first on their CUs in the same order, and nothing is left to even things out.
// With the heaviest first throughout, the heaviest CU of a causal launch holds tile 0 and
// the middle one; so the second 256 run lightest first (`n` items, `first` on the CUs
// before the second round starts). On MI355X, causal, us before / after: fp32 forward B 2,
// 8 heads, S 1024, D 64 38.5 / 33.8, B 1, 8, 2000 64.5 / 53.1 (their backward, dQ paired,
// 111 / 106, 203 / 186); bf16 forward B 4, 8, 2048, D 128, softcap 57.5 / 53.7, without
// 47.4 / 46.1, D 64 22.3 / 21.7. The bf16 backward kernels did not change.
constexpr int paired_rank(int k, int first, int n) { return k < first ? k : n - 1 - (k - first); }
constexpr int kPaired = 256;  // flag in xcd_group: pair the ranks of each XCD's 32 CUs

// Whether a 16-bit prefill launch may pair its tiles. Not at head_dim 32 (three workgroups
// on a CU), whose launches it slows: 1-4 % at every size without softcap (8 heads, S 8192
// 68.9 / 72.0 us; 32, 2048 21.2 / 21.7), with softcap by up to 1.5 % to 384 workgroups (8,
// S 5120 71.1 / 72.1); past them it gains 4-15 % there (8, S 8192 130 / 113). head_dim 64
// without softcap, also three on a CU, gains up to 4 % (64, 1024 17.5 / 16.8).
constexpr bool prefill_pairs(int head_dim, bool softcap, int64_t grid) {
  return head_dim > 32 ? head_dim <= 192 : softcap && grid > 384;
}

// Prefill: grid = n_units * n_qt workgroups, unit = batch x q-head, jq = query tile
// (jq = 0 is the heaviest causal tile). With xcd_group = G > 0 (needs n_units % 8 ==
// 0), XCD x owns units [x HX, (x + 1) HX) (HX = n_units / 8) and runs them one after
// another, heaviest tile first, except its last min(HX, G) units, whose tiles run
// interleaved (tile j of each in turn), so the launch ends on light tiles instead of
// the last unit's heaviest tiles starting near the end. Without a group, xcd_remap
// (needs grid % 8 == 0) places consecutive ids on one XCD; otherwise ids map in order.
constexpr void prefill_work_item(int bid, int grid, int n_qt, int xcd_group, int xcd_remap,
                                 int& unit, int& jq) {
  if (xcd_group > 0) {
    const int hx = (grid / n_qt) >> 3;
    const int x = bid & 7;
    const int k = (xcd_group & kPaired) ? paired_rank(bid >> 3, 32, grid >> 3) : bid >> 3;
    xcd_group &= kPaired - 1;
    const int gl = hx < xcd_group ? hx : xcd_group;
    const int k0 = (hx - gl) * n_qt;  // tiles of the units run one after another
    if (k < k0) {
      const int u = k / n_qt;
      unit = x * hx + u;
      jq = k - u * n_qt;
    } else {
      const int r = k - k0;
      jq = r / gl;
      unit = x * hx + (hx - gl) + (r - jq * gl);
    }
    return;
  }
  if (xcd_remap) {
    const int per_xcd = grid >> 3;
    bid = (bid & 7) * per_xcd + (bid >> 3);
  }
  unit = bid / n_qt;
  jq = bid - unit * n_qt;
}

// The prefill launcher's choice: causal grids (whose tiles differ in weight) with
// n_units % 8 == 0 interleave the last units of each XCD: all of them when an XCD has at
// most 8 (cfg3 and cfg5: 64 units), else the last four for units of at most 32 tiles
// (cfg2) and the last two for longer ones (the north star). On MI355X, over unit after
// unit: +2-3 % at S = 8192 and +4-8 % at S = 4096 for the last two; then all 8 +2 % at
// cfg3 and +3.5 % at cfg5, the last four +1.5 % at cfg2 (-0.5 % at the north star,
// all 16 there -2.6 %). Other grids that split evenly over the XCDs keep consecutive
// ids on one XCD.
// two_per_cu: the kernel runs two workgroups on a CU; then launches that fit the chip at
// once pair their tiles (all units interleaved: tile rank = position), from eight tiles a
// unit on (below that they differ too little: four tiles 22.7 / 23.1 us).
constexpr void prefill_grid_order(bool causal, int64_t n_units, int64_t grid, int& xcd_group,
                                  int& xcd_remap, bool two_per_cu = false) {
  xcd_remap = (grid % 8 == 0) ? 1 : 0;
  const int64_t n_qt = n_units > 0 ? grid / n_units : 0;
  xcd_group = (causal && n_units % 8 == 0) ? (n_units / 8 <= 8 ? 8 : (n_qt <= 32 ? 4 : 2)) : 0;
  if (two_per_cu && xcd_group == 8 && n_qt >= 8 && grid > 256 && grid <= 512) xcd_group |= kPaired;
}

// The backward's dK/dV and dQ grids (unit = batch x head, tile j = 0 the heaviest causal
// tile) use the same map and the same launcher choice as the prefill.

}  // namespace ffa
