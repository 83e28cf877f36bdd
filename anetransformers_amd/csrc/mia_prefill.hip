// mia_prefill.hip -- the prefill layer's row kernels around its GEMMs
// (mistral/mistral_ane_prefill.h:1081-1110): RMSNorm of the token rows
// (:163-175) and the split of fp32 activations into the GEMM's fp16 planes.
#include <algorithm>

#include "mia_device.h"
#include "mia_kernels.h"

namespace mia {
namespace {

// One workgroup per token row: ss = sum(x^2), scale = 1 / sqrt(ss / dim + eps),
// out = (x * scale) * w, the reference's two roundings (vsmul then vmul).
// The GEMM's fp32 activations as fp16 hi + lo planes (x = hi + lo to ~2^-22:
// hi = fp16(x), lo = fp16(x - hi), both rounded to nearest even), split once
// per GEMM input instead of once per column tile of the GEMM.
__global__ __launch_bounds__(256) void split_hilo_kernel(const float *__restrict__ x, long n8,
                                                         _Float16 *__restrict__ hi,
                                                         _Float16 *__restrict__ lo) {
#pragma clang fp contract(off)
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n8; i += (long)gridDim.x * 256) {
    const f4 a = reinterpret_cast<const f4 *>(x)[2 * i];
    const f4 b = reinterpret_cast<const f4 *>(x)[2 * i + 1];
    h8 vh, vl;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = e < 4 ? a[e] : b[e - 4];
      const _Float16 h = (_Float16)v;
      vh[e] = h;
      vl[e] = (_Float16)(v - (float)h);
    }
    reinterpret_cast<h8 *>(hi)[i] = vh;
    reinterpret_cast<h8 *>(lo)[i] = vl;
  }
}

// With hi set, the normalised rows go out as the Q4_0 GEMM's fp16 hi + lo
// planes (split exactly as split_hilo_kernel does) instead of fp32 to out.
// 512 threads; thread t sums the 4-value groups at 4t + 2048k in k order, then
// the wave sums and their fixed combination: the order the Q4_0 matvec's
// RMSNorm prologue reproduces.
__global__ __launch_bounds__(512) void rmsnorm_kernel(float *out, const float *in, const float *w,
                                                      int dim, float eps, _Float16 *hi,
                                                      _Float16 *lo) {
#pragma clang fp contract(off)
  __shared__ float red[8];
  const int t = blockIdx.x, tid = threadIdx.x;
  const float *x = in + (size_t)t * dim;
  float ss = 0.0f;
  for (int i = 4 * tid; i < dim; i += 4 * 512) {
    const f4 v = *reinterpret_cast<const f4 *>(x + i);
    ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  ss = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
  const float scale = 1.0f / sqrtf(ss / (float)dim + eps);
  const size_t row = (size_t)t * dim;
  for (int i = 4 * tid; i < dim; i += 4 * 512) {
    const f4 v = *reinterpret_cast<const f4 *>(x + i);
    const f4 wv = *reinterpret_cast<const f4 *>(w + i);
    f4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (v[e] * scale) * wv[e];
    if (hi != nullptr) {
      h4 vh, vl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const _Float16 h = (_Float16)r[e];
        vh[e] = h;
        vl[e] = (_Float16)(r[e] - (float)h);
      }
      *reinterpret_cast<h4 *>(hi + row + i) = vh;
      *reinterpret_cast<h4 *>(lo + row + i) = vl;
    } else {
      *reinterpret_cast<f4 *>(out + row + i) = r;
    }
  }
}

}  // namespace

hipError_t launch_split_hilo(const float *x, long n, _Float16 *hi, _Float16 *lo, int num_cus,
                             hipStream_t s) {
  if (n % 8) return hipErrorInvalidValue;
  const long n8 = n / 8;
  const long wgs = std::min<long>((n8 + 255) / 256, 8L * num_cus);
  hipLaunchKernelGGL(split_hilo_kernel, dim3((unsigned)std::max<long>(wgs, 1)), dim3(256), 0, s,
                     x, n8, hi, lo);
  return hipGetLastError();
}

hipError_t launch_rmsnorm(float *out, const float *in, const float *w, int dim, int S, float eps,
                          hipStream_t s) {
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(S), dim3(512), 0, s, out, in, w, dim, eps,
                     (_Float16 *)nullptr, (_Float16 *)nullptr);
  return hipGetLastError();
}

hipError_t launch_rmsnorm_split(_Float16 *hi, _Float16 *lo, const float *in, const float *w,
                                int dim, int S, float eps, hipStream_t s) {
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(S), dim3(512), 0, s, (float *)nullptr, in, w, dim, eps,
                     hi, lo);
  return hipGetLastError();
}

}  // namespace mia
