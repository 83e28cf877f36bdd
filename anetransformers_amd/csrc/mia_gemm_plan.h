// mia_gemm_plan.h -- the tile and the K split of a prefill GEMM launch
// (mia_gemm.hip), host code only: also compiled by the test that pins which
// tiles the GPU tests' shapes reach.
#pragma once
#include <algorithm>
#include <cmath>

#include "mia_kernels.h"

namespace mia {

constexpr int kGemmRows = 256;  // weight rows per workgroup

// Sets tm and ksplit from N, K, S and the kind of weights.  plain: the K split
// by the fixed rule of ks_min alone (sums that are rounded to fp16 and kept, like
// a ring's keys and values, then do not move with the tuning).
//
// 32, 64 or 128 tokens per workgroup, and the K split, by the time they are
// expected to take:
//   - a 64-K stage takes a workgroup `alone` us, or `pair` us while another one is
//     on its CU; a workgroup starts and ends in `ends` us (filling its stages,
//     writing its tile);
//   - with one workgroup to a CU (128 tokens; hi + lo weights) the workgroups run
//     in whole rounds: 280 on 256 CUs take as long as 512.  Of pairs, a last round
//     that is part empty costs `tail` of what is empty on top of its share;
//   - a K split adds the reduction: 4.1 us and its partial products.
// The figures are fitted to 864 shapes (S 2 .. 1024, 4096 for Q4_0; 4096 / 6144 /
// 14336 / 28672 / 1024 x 4096, 4096 x 14336, 2048 x 1024, 512 x 2048, 8192 x 2560;
// weights from HBM) at every tile and split.  Time over that of the best choice,
// mean and worst, without whole rounds and here: Q4_0 1.013, 1.23 and 1.006,
// 1.18; Q4_K 1.027, 1.31 and 1.002, 1.04; fp16 planes 1.036, 1.32 and 1.006,
// 1.11; Q6_K 1.025, 1.24 and 1.000, 1.03; hi + lo planes 1.054, 1.33 and 1.007,
// 1.18.
// Splits stop where a workgroup would have fewer than four stages.  The split
// does not depend on the form of the weights (Q4_0 in tiles or not, Q4_K or
// its fp16 values, Q6_K or its planes), so that the sums are the same.
inline void gemm_plan(GemmParams &p, int num_cus, bool plain) {
  struct Cost {
    double alone[3], pair[3], ends[3], tail;  // [32, 64, 128 tokens]; pair 0: one to a CU
  };
  static const Cost kCost[3] = {
      {{0.511, 0.799, 0.0}, {0.906, 1.403, 0.0}, {1.8, 2.86, 0.0}, 0.103},  // Q4_0
      {{0.53, 0.76, 1.17}, {1.36, 1.52, 0.0}, {3.3, 4.6, 8.6}, 0.25},  // fp16 weights
      {{1.35, 1.9, 2.35}, {0.0, 0.0, 0.0}, {2.7, 4.9, 15.0}, 0.0},     // hi + lo weights
  };
  const int kind = p.src == kGemmQ40Tile || p.src == kGemmQ40 ? 0
                   : p.src == kGemmQ4K || p.src == kGemmF16   ? 1
                                                              : 2;
  const Cost &c = kCost[kind];
  const long n_all = p.K / gemm_k_unit(p.K);
  // A sum's rounding grows with its length: up to this many splits, partial
  // sums are kept short wherever 64-token tiles leave the device unfilled.
  const long tiles64 = (long)((p.N + kGemmRows - 1) / kGemmRows) * ((p.S + 63) / 64);
  int ks_min = 1;
  while (ks_min < 4 && tiles64 * ks_min * 2 <= 2L * num_cus && n_all / (ks_min * 2) >= 8) ks_min *= 2;
  double best = 0.0;
  for (int i = 0; i < (kind == 0 ? 2 : 3); ++i) {
    const int tokens = 32 << i;
    const long tiles = (long)((p.N + kGemmRows - 1) / kGemmRows) * ((p.S + tokens - 1) / tokens);
    for (int ks = ks_min; ks <= (plain ? ks_min : 16); ks *= 2) {
      if (ks > ks_min && n_all / ks < 4) break;
      const double wgs = (double)(tiles * ks) / num_cus;  // per CU
      const double stages = (double)((n_all + ks - 1) / ks);
      double us = c.alone[i] * stages + c.ends[i];
      if (wgs > 1.0 && c.pair[i] == 0.0) {
        us *= std::ceil(wgs);
      } else if (wgs > 1.0) {
        const double pairs = std::max(1.0, wgs / 2);
        us = (pairs + c.tail * (std::ceil(pairs) - pairs)) * (c.pair[i] * stages + c.ends[i]);
      }
      if (ks > 1) us += 4.1 + 1.2e-6 * (double)ks * p.S * p.N;
      if (best == 0.0 || us < best) {
        best = us;
        p.tm = 1 << i;
        p.ksplit = ks;
      }
    }
  }
  // hi + lo planes of few tokens are bound by their 4 bytes a weight, which 32-token
  // tiles in two rounds read faster (14336 x 4096, 33 tokens: 63 us, 80 in one round)
  if (p.src == kGemmF16x2 && p.S <= 64 && p.ksplit <= 4) p.tm = 1;
}

}  // namespace mia
