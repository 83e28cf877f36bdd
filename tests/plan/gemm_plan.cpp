// The GEMM's plan for tests/test_gemm_plan.py, from the library's own source.
#include "../../anetransformers_amd/csrc/mia_gemm_plan.h"

extern "C" void plan(int src, int N, int K, int S, int num_cus, int plain, int *tm, int *ksplit) {
  mia::GemmParams p{};
  p.src = src;
  p.N = N;
  p.K = K;
  p.S = S;
  mia::gemm_plan(p, num_cus, plain != 0);
  *tm = p.tm;
  *ksplit = p.ksplit;
}
