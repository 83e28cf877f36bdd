// mia_decode.hip -- S=1 GQA decode attention for gfx950 (split-K flash-decode).
//
// Replaces mistral/mistral_model.h:362-487 (gqa_attention_neon), and, in the
// fused variant, steps 4-6 of mistral/mistral_model.h:849-863 (RoPE on q/k,
// fp16 round of k/v, ring write at pos % max_seq, attention).
//
// Grid: one workgroup per (kv head, chunk of the window), 8 waves per
// workgroup, all on that head.  Chunk c is the 16-key tiles c, c + nchunk,
// c + 2 nchunk, ... of the window: spread over the whole ring rather than one
// contiguous block, every workgroup draws on all memory channels alike; wave
// w of the workgroup takes every 8th of its chunk's tiles.  The heads of one
// chunk are consecutive workgroups, which the dispatcher spreads over the
// XCDs.  32 chunks at 8 kv heads fill 256 CUs with 8x fewer split-K partials
// than one wave per head and chunk would leave.
//
// Each wave is an independent pipeline over its tiles, held in a ring of
// register buffers so that the next tiles' loads are in flight while one
// tile is computed.  Every load instruction reads 4 rows x 256 B (whole
// 128-byte lines; loads of 16 rows x 64 B each read a measured 6 % slower):
//   scores  v_mfma_f32_16x16x32_f16: A = 16 key rows (lane = key row), from
//           the loaded K rows re-laid through a per-wave LDS tile; B = the
//           G=4 query heads of the group with q split into fp16 hi + lo
//           parts along K (q = hi + lo to ~2^-22), so the scores carry fp32 q
//           accuracy.
//   softmax wave-local online max / sum in the log2 domain.
//   P.V     v_mfma_f32_16x16x16_f16 computing O^T = V^T P^T: the score
//           accumulator layout (lane = 4 keys of one head) is already the B
//           operand layout with keys along K, so P (fp16 hi + lo) never
//           leaves its lane; V^T comes from the 4 loaded V rows of the lane
//           (4 keys x 8 dims) by byte permutes.
// The 8 waves' results merge through LDS into the chunk's partial (m, l, o)
// (the final output when there is one chunk); a second, small kernel does
// the log-sum-exp merge over chunks.
#include "mia_device.h"
#include "mia_kernels.h"
#include "mia_window.h"

namespace mia {

namespace {

using window::G;
using window::kTile;

constexpr int kWaves = 8;         // waves per workgroup, all on one kv head
constexpr int kThreads = 64 * kWaves;
// Register tile buffers per wave.  One: the buffer is refilled while it is
// consumed (K once staged to LDS, V after the P.V MFMAs), so one tile per wave
// is in flight while the current one is processed.  Two buffers kept more
// loads in flight and read the window ~4 % slower.
constexpr int kDepth = 1;
constexpr int kMaxChunks = 256;  // merge capacity per kv head

// MODE: window::kPlain, kFused, one token at p.pos; kPositions: token
// blockIdx.y at p.positions[blockIdx.y] over the ring as it stands (the chunked
// prefill's phase 2), q rotated in-kernel when theta_inv is set.
template <int MODE>
__global__ void __launch_bounds__(kThreads, 1) decode_kernel(DecodeParams p) {
  __shared__ window::Smem<kWaves> sm;

  // This workgroup's token: window, query, output and partial rows.
  int pos = p.pos, win_L = p.L, win_start = p.start;
  const float *q_in = p.q;
  float *out = p.out, *part_o = p.part_o, *part_ml = p.part_ml;
  if (MODE == window::kPositions) {
    const int tok = blockIdx.y;
    pos = p.positions[tok];
    // mistral_model.h:964-967; a negative position has an empty window
    // (pos + 1 is not formed: it would overflow at INT_MAX)
    win_L = pos < 0 ? 0 : (pos < p.max_seq - 1 ? pos + 1 : p.max_seq);
    win_start = pos < 0 ? 0 : (int)(((long)pos + 1 - win_L) % p.max_seq);
    const size_t rows = (size_t)p.n_kv * G;  // query heads
    q_in += (size_t)tok * rows * HD;
    out += (size_t)tok * rows * HD;
    part_o += (size_t)tok * rows * p.nchunk * HD;
    part_ml += (size_t)tok * rows * p.nchunk * 2;
  }
  const int kvh = blockIdx.x % p.n_kv;
  const int chunk = blockIdx.x / p.n_kv;
  window::attend<MODE, kWaves, kDepth>(
      p, sm, pos, win_L, win_start, q_in, nullptr, kvh, chunk,
      [&](int g, int d, float M, float L, float O) {
        if (p.nchunk == 1) {
          // (an empty window, only in kPositions, writes zeros)
          out[((size_t)kvh * G + g) * HD + d] = L > 0.f ? O / L : 0.f;
        } else {
          const size_t row = ((size_t)kvh * p.nchunk + chunk) * G + g;
          part_o[row * HD + d] = O;
          if (d == 0) *reinterpret_cast<float2 *>(part_ml + row * 2) = make_float2(M, L);
        }
      });
}

// Cross-chunk log-sum-exp merge.  Workgroup = (kv head, q head, block of
// kMergeDims dims); thread = (chunk group cg, dim d).  Every load (the chunk
// maxima and sums, and the thread's partial outputs) is issued before the
// first reduction, so the merge costs one memory round trip.  A separate
// launch: the kernel boundary orders the partial writes before these reads.
// 16 dims per workgroup (256 workgroups for 8 kv heads) measured 1.6 %
// faster per decode step than 32 (128 workgroups) and than 8 (512).
constexpr int kMergeDims = 16;

__global__ void __launch_bounds__(256) decode_merge_kernel(DecodeParams p) {
  constexpr int kDW = kMergeDims;      // dims of one workgroup
  constexpr int kCG = 256 / kDW;       // chunk groups (threads per dim)
  constexpr int kPer = kMaxChunks / kCG;  // chunks per thread at most
  __shared__ float mx[8];
  __shared__ float red[kCG][kDW];
  __shared__ float wt[kMaxChunks];
  __shared__ float lsum[8];
  const int db = blockIdx.x % (HD / kDW);
  const int hg = blockIdx.x / (HD / kDW);  // kvh * G + g
  const int kvh = hg / G, g = hg % G;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cg = tid / kDW, d = kDW * db + (tid % kDW);
  // token blockIdx.y (kPositions; 0 otherwise): its partials and output rows
  const size_t tok = blockIdx.y;
  const size_t hb = (size_t)kvh * p.nchunk * G + tok * p.n_kv * p.nchunk * G;
  float2 ml = make_float2(-INFINITY, 0.f);
  if (tid < p.nchunk) ml = *reinterpret_cast<const float2 *>(p.part_ml + (hb + (size_t)tid * G + g) * 2);
  float ov[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = cg + kCG * k;
    ov[k] = c < p.nchunk ? p.part_o[(hb + (size_t)c * G + g) * HD + d] : 0.f;
  }
  // max over chunks
  float m = wave_max(ml.x);
  if (lane == 0) mx[wv] = m;
  __syncthreads();
  float M = mx[0];
#pragma unroll
  for (int k = 1; k < 4; ++k) M = fmaxf(M, mx[k]);
  const float Mu = M == -INFINITY ? 0.f : M;
  const float e = ml.x == -INFINITY ? 0.f : fast_exp2(ml.x - Mu);
  if (tid < kMaxChunks) wt[tid] = e;
  float l = wave_sum(e * ml.y);
  if (lane == 0) lsum[wv] = l;
  __syncthreads();
  float O = 0.f;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = cg + kCG * k;
    if (c < p.nchunk) O = __builtin_fmaf(wt[c], ov[k], O);
  }
  red[cg][tid % kDW] = O;
  __syncthreads();
  if (tid < kDW) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < kCG; ++k) t += red[k][tid];
    const float Ls = lsum[0] + lsum[1] + lsum[2] + lsum[3];
    // (Ls = 0 only for an empty window: zeros)
    p.out[(tok * p.n_kv * G + hg) * HD + d] = Ls > 0.f ? t / Ls : 0.f;
  }
}

}  // namespace

size_t decode_scratch_bytes(int n_kv, int g, int nchunk, int n_tok) {
  return (size_t)n_tok * n_kv * nchunk * g * (HD + 2) * sizeof(float);
}

int decode_pick_nchunk(int L, int n_kv, int target_wgs) {
  const int n_tiles = (L + kTile - 1) / kTile;
  // one workgroup per (kv head, chunk), about target_wgs of them; at least
  // one tile per wave, at most kMaxChunks chunks
  int nchunk = (target_wgs + n_kv - 1) / n_kv;
  const int per_wave = (n_tiles + kWaves - 1) / kWaves;
  if (nchunk > per_wave) nchunk = per_wave;
  if (nchunk > kMaxChunks) nchunk = kMaxChunks;
  if (nchunk < 1) nchunk = 1;
  return nchunk;
}

hipError_t launch_decode(const DecodeParams &p, int g, int mode, hipStream_t s, hipEvent_t ev0,
                         hipEvent_t ev1) {
  if (g != G) return hipErrorInvalidValue;
  if (p.nchunk < 1 || p.nchunk > kMaxChunks) return hipErrorInvalidValue;
  const bool positions = mode == kDecodePositions;
  if (positions && (p.positions == nullptr || p.n_tok < 1 || p.n_tok > 65535))
    return hipErrorInvalidValue;
  dim3 grid(p.n_kv * p.nchunk, positions ? p.n_tok : 1), block(kThreads);
  if (mode == kDecodeFused)
    hipExtLaunchKernelGGL(decode_kernel<window::kFused>, grid, block, 0, s, ev0, ev1, 0, p);
  else if (positions)
    hipExtLaunchKernelGGL(decode_kernel<window::kPositions>, grid, block, 0, s, ev0, ev1, 0, p);
  else
    hipExtLaunchKernelGGL(decode_kernel<window::kPlain>, grid, block, 0, s, ev0, ev1, 0, p);
  return hipGetLastError();
}

hipError_t launch_decode_merge(const DecodeParams &p, hipStream_t s) {
  const int ntok = p.positions != nullptr ? p.n_tok : 1;
  if (p.nchunk > 1)
    hipLaunchKernelGGL(decode_merge_kernel, dim3(p.n_kv * G * (HD / kMergeDims), ntok), dim3(256),
                       0, s, p);
  return hipGetLastError();
}

}  // namespace mia
