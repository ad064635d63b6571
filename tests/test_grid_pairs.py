"""Paired workgroup order of launches that fit the chip at once: a g++ build of ffa_grid.h
checks that the order is one-to-one and that it evens out the load of the CUs."""

from __future__ import annotations

import os
import subprocess

from fastest_flash_attention_amd.kernels.hip import build

SOURCE = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "ffa_grid.h"

int main() {
  int paired = 0, lighter = 0;
  for (int units = 1; units <= 64; ++units) {
    for (int n_t = 1; n_t <= 64; ++n_t) {
      const int grid = units * n_t;
      int group = 0, remap = 0;
      ffa::prefill_grid_order(true, units, grid, group, remap, true);
      if (!(group & ffa::kPaired)) continue;
      if (grid <= 256 || grid > 512) return std::printf("paired grid %d\n", grid), 1;
      ++paired;
      std::vector<int> seen(grid, 0);
      std::vector<long> cu(256, 0), plain(256, 0);
      for (int bid = 0; bid < grid; ++bid) {
        int u = -1, j = -1;
        ffa::prefill_work_item(bid, grid, n_t, group, remap, u, j);
        if (u < 0 || u >= units || j < 0 || j >= n_t || seen[u * n_t + j]++) {
          return std::printf("units %d tiles %d: id %d -> (%d, %d)\n", units, n_t, bid, u, j), 1;
        }
        // CU = XCD (bid % 8), then the XCD's 32 CUs in turn; causal weight of tile j
        const int c = (bid & 7) * 32 + ((bid >> 3) & 31);
        cu[c] += n_t - j;
        ffa::prefill_work_item(bid, grid, n_t, group & (ffa::kPaired - 1), remap, u, j);
        plain[c] += n_t - j;
      }
      const long most = *std::max_element(cu.begin(), cu.end());
      const long before = *std::max_element(plain.begin(), plain.end());
      if (most > before) return std::printf("units %d tiles %d: heavier than unpaired\n", units, n_t), 1;
      lighter += most < before;
      // a full launch: every CU gets the two tiles whose weights add up to n_t + 1
      if (grid == 512 && most > n_t + 1) return std::printf("units %d tiles %d: %ld\n", units, n_t, most), 1;
    }
  }
  for (int n = 257; n <= 512; ++n) {
    std::vector<int> seen(n, 0);
    for (int k = 0; k < n; ++k) {
      const int r = ffa::paired_rank(k, 256, n);
      if (r < 0 || r >= n || seen[r]++) return std::printf("rank %d of %d -> %d\n", k, n, r), 1;
    }
  }
  // head_dim 32 only where pairing is faster: with softcap past 384 workgroups
  for (int d : {8, 16, 32}) {
    if (ffa::prefill_pairs(d, false, 512) || ffa::prefill_pairs(d, true, 384) ||
        !ffa::prefill_pairs(d, true, 385)) {
      return std::printf("head_dim %d\n", d), 1;
    }
  }
  for (int d : {40, 64, 128, 192}) {
    if (!ffa::prefill_pairs(d, false, 257)) return std::printf("head_dim %d\n", d), 1;
  }
  if (ffa::prefill_pairs(200, true, 400)) return std::printf("head_dim 200\n"), 1;
  std::printf("ok %d, %d of them lighter\n", paired, lighter);
  return paired == 0 || 2 * lighter < paired;
}
"""


def test_paired_order(tmp_path):
    src, exe = tmp_path / "pairs.cpp", tmp_path / "pairs"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{build.HERE}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert r.stdout.startswith("ok")
