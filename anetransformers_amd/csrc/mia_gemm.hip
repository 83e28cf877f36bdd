// mia_gemm.hip -- the prefill GEMMs (mistral/mistral_ane_prefill.h:999-1042;
// the reference dequantises 128-row weight tiles to fp32 and calls
// cblas_sgemm), with epilogues for the residual adds and SwiGLU
// (mistral_model.h:174-199).
//
// Y[S][N] = X[S][K] . W[N][K]^T on fp16 MFMA (v_mfma_f32_32x32x16_f16) with
// fp32 accuracy where it matters: X comes as fp16 hi + lo planes (x = hi + lo
// to ~2^-22, split by its producer) and both halves go through the MFMA.  The
// weights enter as fp16 operands that are exact or carry 22 bits:
//   Q4_0   q - 8 (exact); the fp16 block scale d is applied in fp32 once per
//          32-value block, acc += d * (X . q), which is what dequantising to
//          fp32 computes
//   Q4_K   the reference's weights are fp16 values (dequant_q4_K_block_neon,
//          dequant.h:68-125), formed in registers by its fp16 steps
//   F16    fp16 values; also Q4_K weights written out once at load time
//   Q6_K, F32   row-scaled fp16 hi + lo halves, a third MFMA for X's hi part
//          against the lo half, the row scale at the end: planes written by
//          launch_typed_split, or the same halves formed in registers from
//          Q6_K blocks regrouped by launch_q6k_regroup (a byte per weight
//          instead of four)
//
// Workgroup: 256 threads, 32 TM tokens x 256 weight rows.  Wave w owns 64
// weight rows (two 32-row MFMA tiles) against all tokens, so a weight is
// turned into its fp16 operand once per 32 TM tokens, in the registers of the
// wave that uses it.  Everything arrives in LDS by direct loads
// (global_load_lds), three or four stages deep, one barrier per stage:
//   - the activations' hi and lo planes, shared by the four waves, swizzled so
//     that operand reads are conflict-free;
//   - each wave's own weight rows, read back by that wave alone.
// The K loop is pipelined by hand in steps of 16 K values (Q4_0: 32, a block):
// while the MFMAs of a step run, the next step's activation operands are read
// from LDS, its weights are dequantised, and Q4_0's block scales of the tile
// before are applied, in fenced slots of one MFMA each (a wave issues in
// order, so VALU work has to stand between MFMAs to run under them).
#include <type_traits>

#include "mia_device.h"
#include "mia_gemm_plan.h"
#include "mia_kernels.h"

namespace mia {
namespace {

constexpr int kGThreads = 256;
constexpr int kWN = kGemmRows;  // weight rows per workgroup
constexpr int kQBK = 64;    // K values of a Q4_0 tile column, and of a stage of quantised weights
constexpr int kQ4KBytes = 144;  // a Q4_K block of 256 weights

// The GEMM tile layout of a Q4_0 matrix [N][K / 32 blocks], N and K multiples
// of 64: tile (s, i) holds rows 64 s .. 64 s + 63 and blocks 2 i, 2 i + 1 at
// byte (s * (K / 64) + i) * 2304:
//   - bytes h * 1024 + rr * 16 + 8 * bb + j (half h, row rr, block bb, j < 8):
//     byte 8 h + kPackOrder[j] of the block's 16 quant bytes;
//   - bytes 2048 + rr * 4 + 2 * bb: the block's fp16 scale.
// A wave stages its rows with two 16-byte and one 4-byte direct load per
// lane, and a lane (row rr, half h) reads its 16 quant bytes in one 16-byte
// LDS read.  In each 4 bytes the order 0, 2, 1, 3 puts the quant bytes of a
// value pair (2t, 2t + 1) in bytes 0 and 2 (t even) or 1 and 3 (t odd), so a
// shift and a mask give both values' nibbles under the fp16 exponent.
constexpr int kPackTile = 2304;
__device__ constexpr int kPackOrder[8] = {0, 2, 1, 3, 4, 6, 5, 7};

template <int SRC, int TM>
struct GemmLay {
  static constexpr bool kHalves = SRC == kGemmF16 || SRC == kGemmF16x2;  // fp16 planes
  static constexpr bool kLo = SRC == kGemmF16x2 || SRC == kGemmQ6K;  // hi + lo weights
  static constexpr bool kScaled = SRC == kGemmQ40Tile || SRC == kGemmQ40;
  static constexpr int kBK = kHalves ? 32 : kQBK;   // K values per stage
  static constexpr int kRow = kBK * 2;              // bytes of a plane's row in a stage
  static constexpr int kPlane = 32 * TM * kRow;     // one activation plane
  static constexpr int kBPlane = 64 * kRow;         // one wave's rows of a weight plane
  // one wave's weight rows
  static constexpr int kBWave = SRC == kGemmF16     ? kBPlane
                                : SRC == kGemmF16x2 ? 2 * kBPlane
                                : SRC == kGemmQ4K   ? 64 * 32
                                : SRC == kGemmQ6K   ? 64 * 64
                                                    : 64 * 36;
  static constexpr int kStage = 2 * kPlane + 4 * kBWave;
  // Q4_K: the blocks' 16-byte headers apart, two blocks (of four stages each) deep
  static constexpr int kHdr = SRC == kGemmQ4K ? 4 * 64 * 16 : 0;
  // direct loads per wave and stage
  static constexpr int kALoads = 2 * kPlane / 4096;
  static constexpr int kBLoads = SRC == kGemmQ40  ? 9
                                 : kHalves || SRC == kGemmQ6K ? kBWave / 1024
                                                  : 3;
  static constexpr int kLoads = kALoads + kBLoads;
  // workgroups that share a CU (registers, and its 160 KB of LDS), and the
  // stages in flight: three, or four where they fit
  static constexpr int kPerCU = TM <= 2 && 2 * (3 * kStage + 2 * kHdr) <= 160 * 1024 ? 2 : 1;
  static constexpr int kStages = kHalves && kPerCU * 4 * kStage <= 160 * 1024 ? 4 : 3;
  static constexpr int kBytes = kStages * kStage + 2 * kHdr;
};

// Chunk swizzle of a 128-byte activation row r: rows r and r + 8 (same bank
// half, same r & 7) get different chunks, so 16 rows read together hit 16
// different 16-byte bank groups, 8 rows 8 different ones.
// 64-byte rows: four rows cover the banks, rows r, r + 4, r + 8, r + 12 get
// different chunks.
template <int ROW>
__device__ __forceinline__ int aswz(int r) {
  static_assert(ROW == 128 || ROW == 64, "stages of 64 or 32 K values");
  return ROW == 128 ? (r & 7) ^ ((r >> 3) & 1) : (r >> 2) & 3;
}

// Direct loads from global memory into LDS, 16 (dwordx4) or 4 (dword) bytes per
// lane at byte M0 + offset + lane * size: the immediate offset applies to both
// addresses, so a group of loads shares one M0 and each address carries minus
// its offset.  Completion is awaited with vmcnt (the compiler does not track
// these loads).
//   activations: N loads of 1 KB, lane address base + off[j] (off[] with
//   1024 j taken off and kBias added, base with kBias taken off, so that no
//   32-bit offset is negative)
constexpr unsigned kBias = 4096;
template <int N>
__device__ __forceinline__ void dma_planes(const void *base, const unsigned *off, unsigned m) {
  static_assert(N == 1 || N == 2 || N == 4, "one, two or four loads per M0");
  if constexpr (N == 1)
    asm volatile(
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %0"
        ::"s"(base), "v"(off[0]), "s"(m)
        : "memory");
  else if constexpr (N == 2)
    asm volatile(
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %0\n\t"
        "global_load_lds_dwordx4 %2, %0 offset:1024"
        ::"s"(base), "v"(off[0]), "v"(off[1]), "s"(m)
        : "memory");
  else
    asm volatile(
        "s_mov_b32 m0, %5\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %0\n\t"
        "global_load_lds_dwordx4 %2, %0 offset:1024\n\t"
        "global_load_lds_dwordx4 %3, %0 offset:2048\n\t"
        "global_load_lds_dwordx4 %4, %0 offset:3072"
        ::"s"(base), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(m)
        : "memory");
}
//   a wave's 2,304 bytes of Q4_0 tiles
__device__ __forceinline__ void dma_q4_tile(const void *a, const void *b, const void *c,
                                            unsigned m) {
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off\n\t"
      "global_load_lds_dwordx4 %1, off offset:1024\n\t"
      "global_load_lds_dword %2, off offset:2048"
      ::"v"(a), "v"(b), "v"(c), "s"(m)
      : "memory");
}
//   three dword loads, 256 bytes apart in LDS
__device__ __forceinline__ void dma_dwords3(const void *a, const void *b, const void *c,
                                            unsigned m) {
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %0, off\n\t"
      "global_load_lds_dword %1, off offset:256\n\t"
      "global_load_lds_dword %2, off offset:512"
      ::"v"(a), "v"(b), "v"(c), "s"(m)
      : "memory");
}
//   32 rows x 32 bytes twice at m, 64 headers at mh
__device__ __forceinline__ void dma_q4k(const void *a, const void *b, const void *h, unsigned m,
                                        unsigned mh) {
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off\n\t"
      "global_load_lds_dwordx4 %1, off offset:1024\n\t"
      "s_mov_b32 m0, %4\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, off"
      ::"v"(a), "v"(b), "v"(h), "s"(m), "s"(mh)
      : "memory");
}
//   four 1 KB pieces of a weight plane
__device__ __forceinline__ void dma_rows4(const void *a, const void *b, const void *c,
                                          const void *d, unsigned m) {
  asm volatile(
      "s_mov_b32 m0, %4\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off\n\t"
      "global_load_lds_dwordx4 %1, off offset:1024\n\t"
      "global_load_lds_dwordx4 %2, off offset:2048\n\t"
      "global_load_lds_dwordx4 %3, off offset:3072"
      ::"v"(a), "v"(b), "v"(c), "v"(d), "s"(m)
      : "memory");
}
template <int N>
__device__ __forceinline__ void gemm_wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ float f16_bits_f32(unsigned h) {
  return (float)__builtin_bit_cast(_Float16, (unsigned short)(h & 0xFFFFu));
}

typedef __attribute__((address_space(3))) h8 lds_h8;
typedef __attribute__((address_space(3))) u4 lds_u4;
typedef __attribute__((address_space(3))) unsigned lds_u32;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h8 lds_read_h8(unsigned a) { return *(const lds_h8 *)(__UINTPTR_TYPE__)a; }
__device__ __forceinline__ u4 lds_read_u4(unsigned a) { return *(const lds_u4 *)(__UINTPTR_TYPE__)a; }
__device__ __forceinline__ unsigned lds_read_u32(unsigned a) {
  return *(const lds_u32 *)(__UINTPTR_TYPE__)a;
}

// gate * sigmoid(gate) * up (silu_mul_neon, mistral_model.h:174-199)
__device__ __forceinline__ float silu_mul(float g, float u) {
#pragma clang fp contract(off)
  const float sig = 1.0f / (1.0f + expf(-g));
  return (g * sig) * u;
}

// Element (m, n) of the product, v (kGemmStore, kGemmAdd).
template <int MODE>
__device__ __forceinline__ void gemm_epilogue(const GemmParams &p, int m, int n, float v) {
  if (MODE == kGemmStore) {
    if (n < p.rows0)
      p.y0[(size_t)m * p.rows0 + n] = v;
    else if (n < p.rows01)
      p.y1[(size_t)m * (p.rows01 - p.rows0) + (n - p.rows0)] = v;
    else
      p.y2[(size_t)m * (p.N - p.rows01) + (n - p.rows01)] = v;
  } else {
    float *y = p.y0 + (size_t)m * p.N + n;
    *y = *y + v;
  }
}

// The SwiGLU product r of token m, hidden unit n as the next GEMM's planes.
__device__ __forceinline__ void swiglu_out(const GemmParams &p, int m, int n, float r) {
  const size_t i = (size_t)m * p.rows0 + n;
  const _Float16 h = (_Float16)r;
  p.ohi[i] = h;
  p.olo[i] = (_Float16)(r - (float)h);
}

// Tile of workgroup L.  The dispatcher hands workgroup L of a launch to XCD
// L mod 8, and each XCD has its own L2.  Without a K split, weight-row tiles
// run fastest (with 8 | nx every XCD keeps its own row tiles: each weight
// byte is fetched into one L2, the activations into all eight).  With a K
// split, workgroup L takes tile w, XCD g owning the contiguous range of w from
// g * T / 8 (T tiles in all; the first T mod 8 XCDs one more), and w runs over
// the token tiles first, then the weight-row tiles, then the splits: an XCD
// works on whole weight-row tiles of one split, and a token tile's
// activations of a split are fetched by the 8 / splits XCDs of that split
// instead of by all eight.
__device__ __forceinline__ void gemm_tile_of(int L, int nx, int ny, int nz, int &tx, int &ty,
                                             int &tz) {
  if (nz == 1) {
    tx = L % nx;
    ty = L / nx;
    tz = 0;
    return;
  }
  const int T = nx * ny * nz;
  const int g = L & 7, j = L >> 3;
  const int wi = g * (T >> 3) + min(g, T & 7) + j;
  ty = wi % ny;
  const int r = wi / ny;
  tx = r % nx;
  tz = r / nx;
}

template <int MODE, int SRC, int TM>
__global__ __launch_bounds__(kGThreads, (GemmLay<SRC, TM>::kPerCU)) void gemm_kernel(GemmParams p) {
#pragma clang fp contract(off)
  using L = GemmLay<SRC, TM>;
  constexpr int kBK = L::kBK;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  int tx, ty, tz;
  gemm_tile_of(blockIdx.x, (p.N + kWN - 1) / kWN, (p.S + 32 * TM - 1) / (32 * TM), p.ksplit, tx,
               ty, tz);
  const int m0 = ty * 32 * TM;
  // first column of the wave: of the product, or (SwiGLU) of the hidden units
  const int nw = MODE == kGemmSwiGlu ? tx * (kWN / 2) + 32 * w : tx * kWN + 64 * w;
  // K in units of gemm_k_unit, split alike for every source
  const int n_units = p.K / gemm_k_unit(p.K), per_unit = gemm_k_unit(p.K) / kBK;
  const int it0 = (int)((long)n_units * tz / p.ksplit) * per_unit;
  const int n_it = (int)((long)n_units * (tz + 1) / p.ksplit) * per_unit - it0;
  const int last = it0 + n_it - 1;
  const unsigned sbase = __builtin_amdgcn_readfirstlane((unsigned)(__UINTPTR_TYPE__)smem);

  // Row v (0 .. 63) of the wave: its matrix and row there.  SwiGLU: 32 gate
  // rows, then the same 32 up rows.  Rows past N load the last row; their
  // results are not written.
  auto row_of = [&](int v, const uint8_t *&base) {
    if (MODE == kGemmSwiGlu) {
      base = v < 32 ? p.w0 : p.w1;
      return min(nw + (v & 31), p.rows0 - 1);
    }
    const int g = min(nw + v, p.N - 1);
    base = g < p.rows0 ? p.w0 : (g < p.rows01 ? p.w1 : p.w2);
    return g < p.rows0 ? g : (g < p.rows01 ? g - p.rows0 : g - p.rows01);
  };

  // Activation loads: wave w fills rows of plane w / 2, kRows rows per load;
  // lane i takes row i / kChunks, LDS chunk i % kChunks.
  constexpr int kChunks = L::kRow / 16, kRows = 64 / kChunks;
  constexpr int kAGroup = L::kALoads < 4 ? L::kALoads : 4;  // loads per M0
  unsigned aoff[L::kALoads];
#pragma unroll
  for (int j = 0; j < L::kALoads; ++j) {
    const int r = 16 * TM * (w & 1) + kRows * j + lane / kChunks;
    const int c = (lane % kChunks) ^ aswz<L::kRow>(r);
    aoff[j] = (unsigned)(min(r, p.S - 1 - m0) * p.K + 8 * c) * 2u + kBias - 1024u * (j % kAGroup);
  }
  const char *const asrc =
      reinterpret_cast<const char *>((w >> 1 ? p.alo : p.ahi) + (size_t)m0 * p.K) - kBias;
  const unsigned a_lds = (unsigned)(w * L::kPlane / 2);
  // Weight loads of the wave's 64 rows:
  //   Q4_0 tiles  two 16-byte loads and one 4-byte load per lane (row = lane)
  //   Q4_0        64 rows x 9 dwords, dword q = 64 j + lane, row q / 9
  //   Q4_K        32 quant bytes per row (lane = 2 row + 16-byte piece), and
  //               the block's header (row = lane)
  //   Q6_K        16 rows x 64 bytes per load, 16-byte pieces swizzled
  //   planes      likewise, as the activations' chunks
  constexpr int kBPtrs = SRC == kGemmQ40 ? 9 : (L::kHalves || SRC == kGemmQ6K ? 4 : 3);
  const uint8_t *bsrc[kBPtrs];
  const size_t lo_plane = SRC == kGemmF16x2 ? p.lo_bytes : 0;
#pragma unroll
  for (int j = 0; j < kBPtrs; ++j) {
    const uint8_t *base;
    if constexpr (SRC == kGemmQ40Tile) {
      const int r = row_of(lane, base);
      const uint8_t *tile = base + (size_t)(r / 64) * (size_t)(p.K / kQBK) * kPackTile;
      bsrc[j] = tile + (j < 2 ? 16 : 4) * (r & 63);  // + 1024 j by the load
    } else if constexpr (SRC == kGemmQ40) {
      const int q = 64 * j + lane;
      const int r = row_of(q / 9, base);
      bsrc[j] = base + (size_t)r * (size_t)(p.K / 32) * 18 + 4 * (q % 9) - 256 * (j % 3);
    } else if constexpr (SRC == kGemmQ4K) {
      const int r = row_of(j < 2 ? 32 * j + (lane >> 1) : lane, base);
      bsrc[j] = base + (size_t)r * (size_t)(p.K / 256) * kQ4KBytes +
                (j < 2 ? 16 + 16 * (lane & 1) - 1024 * j : 0);
    } else {
      const int v = 16 * j + (lane >> 2);
      const int r = row_of(v, base);
      bsrc[j] = base + (size_t)r * p.K * (L::kHalves ? 2 : 1) +
                16 * ((lane & 3) ^ aswz<64>(v)) - 1024 * j;
    }
  }
  const unsigned b_lds = (unsigned)(2 * L::kPlane + w * L::kBWave);
  const unsigned h_lds = sbase + (unsigned)(L::kStages * L::kStage + w * 1024);  // Q4_K headers
  // K block `it` (absolute) into stage slot `st`, in kParts groups of loads.
  constexpr int kAParts = L::kALoads / kAGroup;
  constexpr int kParts = kAParts + (SRC == kGemmQ40 ? 3 : (SRC == kGemmF16x2 ? 2 : 1));
  auto issue_part = [&](int st, int it, int part) {
    const unsigned sb = sbase + (unsigned)(st * L::kStage);
    if (part < kAParts) {
      dma_planes<kAGroup>(asrc + (size_t)(unsigned)it * (kBK * 2), aoff + part * kAGroup,
                          sb + a_lds + 1024u * kAGroup * part);
      return;
    }
    const int b = part - kAParts;
    if constexpr (SRC == kGemmQ40Tile) {
      const unsigned o = (unsigned)it * (unsigned)kPackTile;
      dma_q4_tile(bsrc[0] + o, bsrc[1] + o, bsrc[2] + o, sb + b_lds);
    } else if constexpr (SRC == kGemmQ40) {
      const unsigned o = (unsigned)it * 36u;
      dma_dwords3(bsrc[3 * b] + o, bsrc[3 * b + 1] + o, bsrc[3 * b + 2] + o, sb + b_lds + 768u * b);
    } else if constexpr (SRC == kGemmQ4K) {
      // (the headers come again with every stage of their block, so that
      // every stage issues the same number of loads; a block's header slot is
      // rewritten for the block after the next only once this one is past)
      const unsigned h = (unsigned)(it >> 2) * (unsigned)kQ4KBytes, o = h + 32u * (it & 3);
      dma_q4k(bsrc[0] + o, bsrc[1] + o, bsrc[2] + h, sb + b_lds,
              h_lds + (unsigned)(((it >> 2) & 1) * L::kHdr));
    } else {
      const size_t o = (size_t)(unsigned)it * 64u + (b ? lo_plane : 0);
      dma_rows4(bsrc[0] + o, bsrc[1] + o, bsrc[2] + o, bsrc[3] + o,
                sb + b_lds + (b ? L::kBPlane : 0));
    }
  };
  auto issue = [&](int st, int it) {
#pragma unroll
    for (int i = 0; i < kParts; ++i) issue_part(st, it, i);
  };

  f16v acc[TM][2];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[tm][tn][i] = 0.0f;

  // (opaque, in VGPRs and one in an SGPR: an AND-OR takes no literals)
  unsigned nib_mask = 0x000F000Fu, top_mask = 0x00300030u, nib_exp = 0x64006400u;
  asm volatile("" : "+v"(nib_mask), "+v"(top_mask), "+s"(nib_exp));
  auto fence = [] { __builtin_amdgcn_sched_barrier(0); };

  // Operand (k-step ks of the 32-K block kb) of token row 32 tm + col: the
  // 16-byte chunk 4 kb + 2 ks + half of the row for Q4_0, whose quant bytes
  // pair values 16 apart, and 4 kb + 2 half + ks for the others (a Q4_K lane
  // then holds 16 consecutive quant bytes of its row; the planes take the same
  // order, so that Q4_K weights give the same sums in either form).  The row's
  // swizzle is an XOR of disjoint address bits: per-lane base ^ constant.
  constexpr int kHalfChunk = L::kScaled ? 1 : 2, kStepChunk = L::kScaled ? 2 : 1;
  const unsigned a_lane = (unsigned)(col * L::kRow + 16 * ((kHalfChunk * half) ^ aswz<L::kRow>(col)));
  auto read_a1 = [&](h8 &hi, h8 &lo, unsigned sb, int kb, int ks, int tm) {
    const unsigned ad =
        sb + (a_lane ^ (unsigned)(16 * (4 * kb + kStepChunk * ks))) + (unsigned)(tm * 32 * L::kRow);
    hi = lds_read_h8(ad);
    lo = lds_read_h8(ad + L::kPlane);
  };

  // A stage's weights of the lane's two rows (tn), as they lie in LDS.
  struct BRaw {
    unsigned nb[2][2][2];  // Q4_0: [block][tn][dword], 8 quant bytes
    unsigned s[2][2];      // Q4_0: scale bits [block][tn]
    u4 q[2], hdr[2];       // Q4_K, Q6_K: the lane's 16 low-nibble bytes, and the block
                           // header or the lane's high bits and scales [tn]
  };
  auto read_b = [&](BRaw &b, unsigned sb, int it) {
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) {
      const int rr = 32 * tn + col;
      if constexpr (SRC == kGemmQ40Tile) {
        const u4 qv = lds_read_u4(sb + b_lds + (unsigned)(half * 1024 + rr * 16));
        const unsigned s = lds_read_u32(sb + b_lds + (unsigned)(2048 + rr * 4));
        b.nb[0][tn][0] = qv[0];
        b.nb[0][tn][1] = qv[1];
        b.nb[1][tn][0] = qv[2];
        b.nb[1][tn][1] = qv[3];
        b.s[0][tn] = s;
        b.s[1][tn] = s >> 16;
      } else if constexpr (SRC == kGemmQ40) {
        // dwords 2h .. 2h+2 (block 0's nibbles 8h .. 8h+7 at byte offset 2),
        // dword 0 (scale 0, low half), dword 4 (scale 1, high half), dwords
        // 5+2h, 6+2h (block 1's nibbles 8h .. 8h+7)
        const unsigned rb = sb + b_lds + (unsigned)(rr * 36);
        const unsigned rh = rb + 8u * half;
        const unsigned x0 = lds_read_u32(rh), x1 = lds_read_u32(rh + 4), x2 = lds_read_u32(rh + 8);
        b.nb[0][tn][0] = __builtin_amdgcn_alignbyte(x1, x0, 2);
        b.nb[0][tn][1] = __builtin_amdgcn_alignbyte(x2, x1, 2);
        b.nb[1][tn][0] = lds_read_u32(rh + 20);
        b.nb[1][tn][1] = lds_read_u32(rh + 24);
        b.s[0][tn] = lds_read_u32(rb);
        b.s[1][tn] = lds_read_u32(rb + 16) >> 16;
      } else if constexpr (SRC == kGemmQ4K) {
        b.q[tn] = lds_read_u4(sb + b_lds + (unsigned)(rr * 32 + half * 16));
        b.hdr[tn] = lds_read_u4(h_lds + (unsigned)(((it >> 2) & 1) * L::kHdr + rr * 16));
      } else if constexpr (SRC == kGemmQ6K) {
        const unsigned rb = sb + b_lds + (unsigned)(rr * 64);
        b.q[tn] = lds_read_u4(rb + 16u * (half ^ aswz<64>(rr)));
        b.hdr[tn] = lds_read_u4(rb + 16u * ((2 + half) ^ aswz<64>(rr)));
      }
    }
  };
  // Block kb's scales of the lane's two rows: Q4_0 d, Q4_K the sub-block scale
  // and min (both halves).
  struct BScale {
    float d[2];
    h2 vd[2], vm[2];
  };
  auto scales = [&](BScale &o, const BRaw &b, int kb, int it) {
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) {
      if constexpr (L::kScaled) {
        o.d[tn] = f16_bits_f32(b.s[kb][tn]);
        // converted once here: folded into each FMA, the conversion makes
        // every scale FMA a mixed-precision one
        asm volatile("" : "+v"(o.d[tn]));
      } else if constexpr (SRC == kGemmQ4K) {
        // get_scale_min_k4 (dequant.h:58-66) of sub-block j: its bytes sit at
        // position j % 4 of the words holding scale bytes 0-3, 4-7 and 8-11
        const int j = 2 * (it & 3) + kb;
        const unsigned e0 = b.hdr[tn].x, e1 = b.hdr[tn].y, e2 = b.hdr[tn].z, e3 = b.hdr[tn].w;
        const int p8 = 8 * (j & 3);
        const unsigned x1 = e1 >> p8, x2 = e2 >> p8, x3 = e3 >> p8;
        const unsigned late = j < 4 ? 0u : ~0u;  // (masks: a branch would split the step)
        const unsigned sv = (x1 & 63 & ~late) | (((x3 & 0xF) | ((x1 >> 2) & 0x30)) & late);
        const unsigned mv = (x2 & 63 & ~late) | ((((x3 >> 4) & 0xF) | ((x2 >> 2) & 0x30)) & late);
        const _Float16 vd = (_Float16)(f16_bits_f32(e0) * (float)sv);
        const _Float16 vm = (_Float16)(f16_bits_f32(e0 >> 16) * (float)mv);
        o.vd[tn] = (h2){vd, vd};
        o.vm[tn] = (h2){vm, vm};
        asm volatile("" : "+v"(o.vd[tn]), "+v"(o.vm[tn]));
      }
    }
  };
  // Operand dword q of (ks, tn) of block kb: two consecutive values.  Their
  // quant bytes go to the two halves of a dword (one byte permute; Q4_0 tiles:
  // a shift, the pair being in bytes 0 and 2 or 1 and 3 already), and one
  // AND-OR leaves the nibbles under the fp16 exponent of 1024 (0x6400 | n =
  // 1024 + n).  Q4_0: the low nibbles are k-step 0, the high ones k-step 1,
  // and subtracting 1032 gives n - 8.  Q4_K: the low nibbles are block 0, the
  // high ones block 1, and w = fl16(fl16(n * vd) - vm).  Q6_K: as Q4_K, with
  // the pair's two top bits each ORed in; ol gets the lo halves.
  auto dequant = [&](u4 &o, u4 &ol, const BRaw &b, const BScale &sc, int kb, int ks, int tn, int q) {
    if constexpr (!L::kHalves) {
      unsigned t;
      if constexpr (SRC == kGemmQ40Tile) {
        t = b.nb[kb][tn][q >> 1] >> (8 * (q & 1) + 4 * ks);
      } else {
        const unsigned x = SRC == kGemmQ40 ? b.nb[kb][tn][q >> 1] : b.q[tn][2 * ks + (q >> 1)];
        const unsigned y = (SRC == kGemmQ40 ? ks : kb) ? x >> 4 : x;
        t = __builtin_amdgcn_perm(y, y, (q & 1) ? 0x0C030C02u : 0x0C010C00u);
      }
      unsigned e = (t & nib_mask) | nib_exp;
      if constexpr (SRC == kGemmQ6K) {
        const unsigned top = b.hdr[tn][kb];  // pair 4 ks + q at bits 2 (4 ks + q) of each half
        const int sh = 2 * (4 * ks + q) - 4;
        e |= (sh >= 0 ? top >> sh : top << -sh) & top_mask;
      }
      const _Float16 zero = (_Float16)(L::kScaled ? 1032.0f : (SRC == kGemmQ6K ? 1056.0f : 1024.0f));
      h2 r = __builtin_bit_cast(h2, e) - (h2){zero, zero};
      if constexpr (SRC == kGemmQ4K) r = r * sc.vd[tn] - sc.vm[tn];
      if constexpr (SRC == kGemmQ6K) {
        // x = scale * (q - 32), exact in fp32, as hi + lo
        const unsigned sb = b.hdr[tn][2 + kb];
        const float ds = __builtin_bit_cast(float, sb);
        const float x0 = ds * (float)r[0], x1 = ds * (float)r[1];
        r = (h2){(_Float16)x0, (_Float16)x1};
        const h2 l = {(_Float16)(x0 - (float)r[0]), (_Float16)(x1 - (float)r[1])};
        const unsigned v = __builtin_bit_cast(unsigned, l);
        asm volatile("" ::"v"(v));
        ol[q] = v;
      }
      const unsigned v = __builtin_bit_cast(unsigned, r);
      asm volatile("" ::"v"(v));  // formed here, not where it is used
      o[q] = v;
    }
  };

  // Slot s holds stage it0 + s (mod kStages).  Loads past the range repeat
  // its last stage (in bounds, into a slot nobody reads), so every stage
  // issues the same number of loads and the waits are exact.
  unsigned sb = sbase, sb_next = sbase + L::kStage;
  int st_load = 0, it_load = 0;  // slot and stage of the loads being issued
  // The next stage's loads are in (this wave's, then everyone's), and everyone
  // has read stage `it` (its operands all come before this point), whose slot
  // takes new loads: they are issued in the slots of the step after this, so
  // that no MFMA waits for them.
  auto advance = [&](int it) {
    gemm_wait_vmcnt<(L::kStages - 2) * L::kLoads>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    it_load = min(it + L::kStages, last);
  };
  auto next_slot = [&] {
    st_load = st_load == L::kStages - 1 ? 0 : st_load + 1;
    sb = sb_next;
    sb_next = sb_next == sbase + (L::kStages - 1) * L::kStage ? sbase : sb_next + L::kStage;
  };
#pragma unroll
  for (int i = 0; i < L::kStages - 1; ++i) issue(i, min(it0 + i, last));
  gemm_wait_vmcnt<(L::kStages - 2) * L::kLoads>();
  asm volatile("s_barrier" ::: "memory");
  issue(L::kStages - 1, min(it0 + L::kStages - 1, last));

  if constexpr (L::kScaled) {
    // Steps of 32 K values, a weight block each: the MFMAs of (a, b), tile by
    // tile (tn, tm), four to a tile's block product, while the next step's
    // operands are formed: activations (na) from block nkb of the stage in
    // slot sb_next, weights (nb) from raw.
    struct AOp {
      h8 hi[2][TM], lo[2][TM];  // [ks][tm]
    };
    struct BOp {
      u4 v[2][2];  // [ks][tn]
      BScale sc;
    };
    f16v blk[2];
    float dprev = 0.0f;
    auto step = [&](const AOp &a, const BOp &b, AOp &na, BOp &nb, const BRaw &raw,
                    unsigned sb_next, int nkb, auto loads) {
      constexpr int kTiles = 2 * TM;
      // First of the next step's 16 operand dwords formed in slot j of tile t.
      auto deq_from = [](int t, int j) {
        if (TM == 2) return 4 * t + (j == 0 ? 0 : (j < 3 ? 2 : j));
        return 8 * t + (j == 0 ? 0 : (j == 1 ? 3 : 2 * j));
      };
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const int tn = t / TM, tm = t % TM;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int ks = j >> 1;
          f16v &c = blk[t & 1];
          const h8 bv = __builtin_bit_cast(h8, b.v[ks][tn]);
          if (j == 0) {
            f16v z;
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = 0.0f;
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi[0][tm], bv, z, 0, 0, 0);
          } else {
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16((j & 1) ? a.lo[ks][tm] : a.hi[ks][tm], bv, c,
                                                       0, 0, 0);
          }
          asm volatile("" : "+v"(c));  // (keeps the MFMA in its slot)
          fence();
          // the tile before: acc += d * block, in the last three slots (its
          // last product is not there yet in the first)
          if (j > 0) {
            const int pn = t > 0 ? (t - 1) / TM : 1, pm = t > 0 ? (t - 1) % TM : TM - 1;
            const float d = t > 0 ? b.sc.d[pn] : dprev;
            const f16v &pb = blk[(t + 1) & 1];
#pragma unroll
            for (int i = j == 1 ? 0 : 5 * j - 4; i < 5 * j + 1; ++i) {
              const float v = __builtin_fmaf(d, pb[i], acc[pm][pn][i]);
              asm volatile("" ::"v"(v));
              acc[pm][pn][i] = v;
            }
          }
          // the next step's activations: a token tile's per tile
          if (j == 0 && t < TM) {
            read_a1(na.hi[0][t], na.lo[0][t], sb_next, nkb, 0, t);
            read_a1(na.hi[1][t], na.lo[1][t], sb_next, nkb, 1, t);
          }
          // and its weights
#pragma unroll
          for (int e = deq_from(t, j); e < deq_from(t, j + 1); ++e)
            dequant(nb.v[e >> 3][(e >> 2) & 1], nb.v[0][0], raw, nb.sc, nkb, e >> 3, (e >> 2) & 1,
                    e & 3);
          if (t == kTiles - 1 && j == 3) scales(nb.sc, raw, nkb, 0);
          if (loads && 4 * t + j >= 1 && 4 * t + j <= kParts) issue_part(st_load, it_load, 4 * t + j - 1);
          fence();
        }
      }
      dprev = b.sc.d[1];
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) blk[1][i] = 0.0f;
    AOp a0, a1;
    BOp b0, b1;
    BRaw r0, r1;
    read_b(r0, sb, it0);
#pragma unroll
    for (int e = 0; e < 2 * TM; ++e)
      read_a1(a0.hi[e / TM][e % TM], a0.lo[e / TM][e % TM], sb, 0, e / TM, e % TM);
    scales(b0.sc, r0, 0, it0);
#pragma unroll
    for (int e = 0; e < 16; ++e)
      dequant(b0.v[e >> 3][(e >> 2) & 1], b0.v[0][0], r0, b0.sc, 0, e >> 3, (e >> 2) & 1, e & 3);
    // (operands formed past the range are a repeated stage's, unused)
    for (int it = it0; it <= last; ++it) {
      step(a0, b0, a1, b1, r0, sb, 1, std::false_type{});
      advance(it);
      read_b(r1, sb_next, it + 1);
      step(a1, b1, a0, b0, r1, sb_next, 0, std::true_type{});
      r0 = r1;
      next_slot();
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      acc[TM - 1][1][i] = __builtin_fmaf(dprev, blk[1][i], acc[TM - 1][1][i]);
  } else {
    // Steps of 16 K values (one MFMA k-step), straight into the accumulators:
    // X's hi part over all tiles, its lo part, and (hi + lo weights) its hi part
    // against the lo half, while the next step's operands arrive.
    constexpr int kPasses = L::kLo ? 3 : 2;
    constexpr int kTiles = 2 * TM, kSlots = kPasses * kTiles;
    struct KOp {
      h8 hi[TM], lo[TM];
      u4 v[2], l[2];  // [tn]; l: the lo half's
    };
    // Planes: operand tn of k-step ks straight from LDS.
    auto read_w = [&](KOp &o, unsigned sb, int ks, int tn) {
      const unsigned ad = sb + b_lds + (a_lane ^ (unsigned)(16 * ks)) + (unsigned)(tn * 32 * L::kRow);
      o.v[tn] = lds_read_u4(ad);
      if constexpr (SRC == kGemmF16x2) o.l[tn] = lds_read_u4(ad + L::kBPlane);
    };
    BScale sc;
    // n: the next step's operands, k-step nk (0 .. kBK / 16 - 1) of stage nit
    // in slot sb_next
    auto step = [&](const KOp &a, KOp &n, const BRaw &raw, unsigned sb_next, int nk, int nit,
                    auto loads) {
      constexpr int kFrom = kSlots / 4;  // first slot with operand dwords
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        const int pass = s / kTiles, tm = s % kTiles / 2, tn = s & 1;
        const h8 av = pass == 1 ? a.lo[tm] : a.hi[tm];
        const h8 bv = __builtin_bit_cast(h8, pass == 2 ? a.l[tn] : a.v[tn]);
        f16v &c = acc[tm][tn];
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, c, 0, 0, 0);
        asm volatile("" : "+v"(c));  // (keeps the MFMA in its slot)
        fence();
        if (s < TM) read_a1(n.hi[s], n.lo[s], sb_next, nk >> 1, nk & 1, s);
        if constexpr (L::kHalves) {
          if (s >= 1 && s < 3) read_w(n, sb_next, nk & 1, s - 1);
        } else {
          if (s == kFrom - 1 && (nk & 1) == 0) scales(sc, raw, nk >> 1, nit);
#pragma unroll
          for (int e = 8 * (s - kFrom) / (kSlots - kFrom);
               s >= kFrom && e < 8 * (s + 1 - kFrom) / (kSlots - kFrom); ++e)
            dequant(n.v[e >> 2], n.l[e >> 2], raw, sc, nk >> 1, nk & 1, e >> 2, e & 3);
        }
        // (after the operand reads, spread where there is room)
        constexpr int kGap = kSlots >= 16 ? 2 : 1;
        if (loads && s >= kSlots - kGap * kParts && (s - (kSlots - kGap * kParts)) % kGap == 0)
          issue_part(st_load, it_load, (s - (kSlots - kGap * kParts)) / kGap);
        fence();
      }
    };
    using F = std::false_type;
    KOp k0, k1;
    BRaw r0, r1;
    read_b(r0, sb, it0);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) read_a1(k0.hi[tm], k0.lo[tm], sb, 0, 0, tm);
    if constexpr (L::kHalves) {
      read_w(k0, sb, 0, 0);
      read_w(k0, sb, 0, 1);
    } else {
      scales(sc, r0, 0, it0);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        dequant(k0.v[e >> 2], k0.l[e >> 2], r0, sc, 0, 0, e >> 2, e & 3);
    }
    // (operands formed past the range are a repeated stage's, unused)
    for (int it = it0; it <= last; ++it) {
      const int nit = min(it + 1, last);
      if constexpr (kBK == 64) {
        step(k0, k1, r0, sb, 1, it, F{});
        step(k1, k0, r0, sb, 2, it, F{});
        step(k0, k1, r0, sb, 3, it, F{});
      } else {
        step(k0, k1, r0, sb, 1, it, F{});
      }
      advance(it);
      read_b(r1, sb_next, nit);
      step(k1, k0, r1, sb_next, 0, nit, std::true_type{});
      r0 = r1;
      next_slot();
    }
  }
  gemm_wait_vmcnt<0>();  // (the repeated loads past the range)
  if constexpr (L::kLo) {
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) {
      const float rs = p.row_scale[min(nw + 32 * tn + col, p.N - 1)];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[tm][tn][i] *= rs;
    }
  }

  // D layout: lane holds column n = col; value i is row 8*(i/4) + 4*half + i%4.
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + 32 * tm + 8 * (i >> 2) + 4 * half + (i & 3);
      if (m >= p.S) continue;
      if (MODE == kGemmSwiGlu) {
        const int n = nw + col;
        if (n >= p.rows0) continue;
        if (p.ksplit > 1) {
          float *pt = p.part + ((size_t)tz * p.S + m) * p.N + n;
          pt[0] = acc[tm][0][i];
          pt[p.rows0] = acc[tm][1][i];
        } else {
          swiglu_out(p, m, n, silu_mul(acc[tm][0][i], acc[tm][1][i]));
        }
      } else {
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
          const int n = nw + 32 * tn + col;
          if (n >= p.N) continue;
          if (p.ksplit > 1)
            p.part[((size_t)tz * p.S + m) * p.N + n] = acc[tm][tn][i];
          else
            gemm_epilogue<MODE>(p, m, n, acc[tm][tn][i]);
        }
      }
    }
  }
}

// Sum of the split partial products in split order, then the epilogue: one
// thread per VEC consecutive columns of a token, span workgroups per token
// (in one grid dimension: the others end at 65,535).
template <int MODE, int VEC>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmParams p, int span) {
  const int m = blockIdx.x / span;
  const int cols = MODE == kGemmSwiGlu ? p.rows0 : p.N;
  const int n = ((int)(blockIdx.x % span) * 256 + threadIdx.x) * VEC;
  if (n >= cols) return;
  const size_t plane = (size_t)p.S * p.N;
  const float *src = p.part + (size_t)m * p.N + n;
  auto sum = [&](const float *s, float (&v)[VEC]) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[e] = 0.0f;
    for (int z = 0; z < p.ksplit; ++z) {
      if constexpr (VEC == 4) {
        const f4 x = *reinterpret_cast<const f4 *>(s + z * plane);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = z == 0 ? x[e] : v[e] + x[e];
      } else {
        v[0] = z == 0 ? s[0] : v[0] + s[z * plane];
      }
    }
  };
  float v[VEC];
  sum(src, v);
  if constexpr (MODE == kGemmSwiGlu) {
    float u[VEC];
    sum(src + p.rows0, u);
#pragma unroll
    for (int e = 0; e < VEC; ++e) swiglu_out(p, m, n + e, silu_mul(v[e], u[e]));
  } else {
#pragma unroll
    for (int e = 0; e < VEC; ++e) gemm_epilogue<MODE>(p, m, n + e, v[e]);
  }
}

// GGUF layout -> GEMM tile layout (above): one thread per (row, block pair),
// 36 bytes in, the same 36 bytes out at their tile places.
__global__ __launch_bounds__(256) void q4_pack_kernel(const uint8_t *__restrict__ src,
                                                      uint8_t *__restrict__ dst, int N, int K) {
  const int steps = K / kQBK;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)N * steps) return;
  const int row = (int)(e / steps), i = (int)(e % steps);
  const unsigned *in = reinterpret_cast<const unsigned *>(src + ((size_t)row * steps + i) * 36);
  unsigned x[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) x[j] = in[j];
  auto byte = [&](int b) { return (x[b >> 2] >> (8 * (b & 3))) & 0xFFu; };
  uint8_t *tile = dst + ((size_t)(row / 64) * steps + i) * kPackTile;
  const int rr = row % 64;
  // block bb: scale at bytes 18 bb, 18 bb + 1; quant bytes at 18 bb + 2 ..
  *reinterpret_cast<unsigned *>(tile + 2048 + 4 * rr) = byte(0) | byte(1) << 8 |
                                                        byte(18) << 16 | byte(19) << 24;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    unsigned o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int bb = d >> 1, j0 = 4 * (d & 1);
      unsigned v = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) v |= byte(18 * bb + 2 + 8 * h + kPackOrder[j0 + j]) << (8 * j);
      o[d] = v;
    }
    *reinterpret_cast<u4 *>(tile + h * 1024 + rr * 16) = (u4){o[0], o[1], o[2], o[3]};
  }
}

template <int MODE, int SRC, int TM>
hipError_t set_lds_limit() {
  return hipFuncSetAttribute((const void *)gemm_kernel<MODE, SRC, TM>,
                             hipFuncAttributeMaxDynamicSharedMemorySize, GemmLay<SRC, TM>::kBytes);
}

template <int MODE, int SRC, int TM>
void launch_tile(const GemmParams &p, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid((unsigned)((p.N + kWN - 1) / kWN * ((p.S + 32 * TM - 1) / (32 * TM)) * p.ksplit));
  hipExtLaunchKernelGGL((gemm_kernel<MODE, SRC, TM>), grid, dim3(kGThreads),
                        (GemmLay<SRC, TM>::kBytes), s, ev0, ev1, 0, p);
}

template <int MODE, int SRC>
void launch_src(const GemmParams &p, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  if (p.tm == 4) {
    if constexpr (!GemmLay<SRC, 1>::kScaled) launch_tile<MODE, SRC, 4>(p, s, ev0, ev1);
  } else if (p.tm == 2) {
    launch_tile<MODE, SRC, 2>(p, s, ev0, ev1);
  } else {
    launch_tile<MODE, SRC, 1>(p, s, ev0, ev1);
  }
}

template <int MODE>
hipError_t launch_mode(const GemmParams &p, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  switch (p.src) {
    case kGemmQ40Tile: launch_src<MODE, kGemmQ40Tile>(p, s, ev0, ev1); break;
    case kGemmQ40: launch_src<MODE, kGemmQ40>(p, s, ev0, ev1); break;
    case kGemmQ4K: launch_src<MODE, kGemmQ4K>(p, s, ev0, ev1); break;
    case kGemmF16: launch_src<MODE, kGemmF16>(p, s, ev0, ev1); break;
    default:
      if constexpr (MODE != kGemmSwiGlu) {
        if (p.rows0 != p.N) return hipErrorInvalidValue;  // one matrix
        if (p.src == kGemmF16x2) launch_src<MODE, kGemmF16x2>(p, s, ev0, ev1);
        else if (p.src == kGemmQ6K) launch_src<MODE, kGemmQ6K>(p, s, ev0, ev1);
        else return hipErrorInvalidValue;
      } else {
        return hipErrorInvalidValue;
      }
  }
  if (p.ksplit > 1) {
    const int cols = MODE == kGemmSwiGlu ? p.rows0 : p.N;
    // four columns per thread where every output row keeps 16-byte steps
    const bool vec = (p.rows0 | p.rows01 | p.N) % 4 == 0;
    const int span = vec ? (cols + 1023) / 1024 : (cols + 255) / 256;
    const dim3 grid((unsigned)span * (unsigned)p.S);
    if (vec)
      hipLaunchKernelGGL((gemm_reduce_kernel<MODE, 4>), grid, dim3(256), 0, s, p, span);
    else
      hipLaunchKernelGGL((gemm_reduce_kernel<MODE, 1>), grid, dim3(256), 0, s, p, span);
  }
  return hipGetLastError();
}

template <int MODE, int SRC>
hipError_t prepare_src() {
  hipError_t e = set_lds_limit<MODE, SRC, 1>();
  if (e == hipSuccess) e = set_lds_limit<MODE, SRC, 2>();
  if constexpr (!GemmLay<SRC, 1>::kScaled)
    if (e == hipSuccess) e = set_lds_limit<MODE, SRC, 4>();
  return e;
}

template <int MODE>
hipError_t prepare_mode() {
  hipError_t e = prepare_src<MODE, kGemmQ40Tile>();
  if (e == hipSuccess) e = prepare_src<MODE, kGemmQ40>();
  if (e == hipSuccess) e = prepare_src<MODE, kGemmQ4K>();
  if (e == hipSuccess) e = prepare_src<MODE, kGemmF16>();
  if constexpr (MODE != kGemmSwiGlu)
    if (e == hipSuccess) e = prepare_src<MODE, kGemmF16x2>();
  if constexpr (MODE != kGemmSwiGlu)
    if (e == hipSuccess) e = prepare_src<MODE, kGemmQ6K>();
  return e;
}

}  // namespace

hipError_t prepare_gemm() {
  const hipError_t e[] = {prepare_mode<kGemmStore>(), prepare_mode<kGemmAdd>(),
                          prepare_mode<kGemmSwiGlu>()};
  for (hipError_t x : e)
    if (x != hipSuccess) return x;
  return hipSuccess;
}

hipError_t launch_gemm(const GemmParams &p, int mode, hipStream_t s, hipEvent_t ev0,
                       hipEvent_t ev1) {
  if (mode == kGemmStore) return launch_mode<kGemmStore>(p, s, ev0, ev1);
  if (mode == kGemmAdd) return launch_mode<kGemmAdd>(p, s, ev0, ev1);
  return launch_mode<kGemmSwiGlu>(p, s, ev0, ev1);
}

hipError_t launch_q4_pack(const void *src, void *dst, int N, int K, hipStream_t s) {
  const long n = (long)N * (K / kQBK);
  hipLaunchKernelGGL(q4_pack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<const uint8_t *>(src), reinterpret_cast<uint8_t *>(dst), N,
                     K);
  return hipGetLastError();
}

}  // namespace mia
