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
// from N, K and S alone, by a fixed rule (sums that are rounded to fp16 and
// kept, like a ring's keys and values, then do not move with the tuning).
// 32, 64 or 128 tokens per workgroup, and the K split, by the time they are
// expected to take (measured over S 8 .. 512 at 4096 / 5120 / 6144 / 28672 x
// 4096 and 4096 x 14336; within 10 % of the best of all the choices there):
//   - a 64-K stage takes a workgroup kAlone us while it has its CU to itself
//     and kShared us of the CU's time when several share it (or follow each
//     other);
//   - a workgroup starts and ends in kEnds us (filling its stages, writing its
//     tile), two of them at a time up to 64 tokens;
//   - a K split adds the reduction: 4 us and reading the partial products at
//     about 6 TB/s (they stay in the caches).
// Splits stop where a workgroup would have fewer than four stages.  The split
// does not depend on the form of the weights (Q4_0 in tiles or not, Q4_K or
// its fp16 values, Q6_K or its planes), so that the sums are the same.
inline void gemm_plan(GemmParams &p, int num_cus, bool plain) {
  // [Q4_0, fp16 weights, hi + lo weights][32, 64, 128 tokens]
  static const double kAlone[3][3] = {{0.62, 1.0, 0.0}, {0.85, 1.1, 1.88}, {1.8, 1.96, 3.0}};
  static const double kShared[3][3] = {{0.56, 0.98, 0.0}, {0.85, 1.2, 1.88}, {1.6, 1.96, 3.0}};
  static const double kEnds[3] = {1.5, 2.5, 5.0};
  const int kind = p.src == kGemmQ40Tile || p.src == kGemmQ40 ? 0
                   : p.src == kGemmQ4K || p.src == kGemmF16   ? 1
                                                              : 2;
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
      const double share = wgs <= 2.0 ? std::ceil(wgs) : wgs + 0.25;
      const double stage =
          share <= 1.0 ? kAlone[kind][i] : std::max(kAlone[kind][i], kShared[kind][i] * share);
      double us = stage * (double)((n_all + ks - 1) / ks) +
                  kEnds[i] * std::ceil(i < 2 ? share / 2 : share);
      if (ks > 1) us += 4.0 + 4e-6 / 6.0 * (double)ks * p.S * p.N;
      if (best == 0.0 || us < best) {
        best = us;
        p.tm = 1 << i;
        p.ksplit = ks;
      }
    }
  }
}

}  // namespace mia
