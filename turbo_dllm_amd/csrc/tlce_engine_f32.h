// 128x128 float32 MFMA tile engine: float32 inputs whose hidden size is a multiple of 4
// (16-byte rows); others take the generic engine.  Cross entropies of some size run on
// the bf16 matrix units instead (tlce_split_f32.h).
//
// Same contract as the other engines: C[i][j] = sum_k A[i][k] * B[j][k] over one tile,
// every product and sum in float32 (v_mfma_f32_16x16x4_f32), operands K-contiguous
// (X[row][k]) or K-major (X[k][row]), any K: what lies past k_end counts as zero.
//
// What bounds it is the float32 matrix rate, 157 TFLOP/s, a sixteenth of bf16's: an MFMA
// occupies its pipe for 32 cycles, so operands are cheap and the tile is small, for its
// tails and its epilogue to overlap: 4 waves of 64x64, two workgroups per CU (64 KiB of
// LDS, at most 256 registers each) of which one computes while the other loads, stores
// or works on its logits.  Operands go global -> VGPR -> LDS one 32-wide K stage ahead
// of two; a K-major operand is transposed in registers, 4x4 elements per thread, so no
// transposed copy of any matrix exists.
//
// LDS stage of one operand: 128 rows x 128 B, 16-byte chunk c (4 K values) of row r in
// slot c ^ ((r >> 1) & 7).  A lane reads one chunk per block and 16-wide K group: lane l
// holds row l%16, K = 4*(l/16) .. +4, and the j-th of four MFMAs takes element j of it.
// Both operands use the same assignment of K values to (lane group, j), and a sum does
// not care which MFMA adds which product.
//
// Measured: 1024 rows, H = 1024, V = 32000, forward and backward in four contractions
// 11.0 -> 2.3 ms (560 to 640 us each, 105 to 120 TFLOP/s; the generic engine reads 17
// LDS words for 16 multiply-adds and reached 20 to 32).
#pragma once

#include "tlce_engine_mfma.h"

namespace tlce {

struct MfmaF32Engine {
  using T = float;
  static constexpr int kTile = 128;
  static constexpr int kThreads = 256;
  static constexpr int kPlanes = 1;
  static constexpr int kWavesPerSimd = 2;
  static constexpr int kBK = 32;
  static constexpr int kTM = 4, kTN = 4;             // 16-row blocks per wave
  static constexpr int kCols = kTN;
  static constexpr int kRows = kTM * 4;
  static constexpr int kShare = 8;
  static constexpr int kOperandBytes = kTile * kBK * 4;        // 16384
  static constexpr int kStageBytes = 2 * kOperandBytes;
  static constexpr int kSmemBytes = 2 * kStageBytes;           // 65536
  static constexpr bool kHasKMajor = true;
  static constexpr bool kPrecise = true;
  static constexpr bool kReadsWhereUsed = false;

  struct Acc { acc4_t c[kTM][kTN]; };

  int lane, wm, wn;

  __device__ __forceinline__ MfmaF32Engine() {
    lane = threadIdx.x & 63;
    wm = threadIdx.x >> 7;
    wn = (threadIdx.x >> 6) & 1;
  }
  __device__ __forceinline__ void forget_lane_invariants() {}
  __device__ __forceinline__ int col(int j) const { return wn * 64 + j * 16 + (lane & 15); }
  __device__ __forceinline__ int row(int i) const {
    return wm * 64 + (i >> 2) * 16 + (lane >> 4) * 4 + (i & 3);
  }
  __device__ __forceinline__ int share_slot() const { return wm * 4 + (lane >> 4); }
  static __device__ __forceinline__ float get(const Acc& a, int j, int i) {
    return a.c[i >> 2][j][i & 3];
  }
  static __device__ __forceinline__ void set(Acc& a, int j, int i, float v) {
    a.c[i >> 2][j][i & 3] = v;
  }
  static __device__ __forceinline__ void zero(Acc& a) {
#pragma unroll
    for (int tm = 0; tm < kTM; ++tm)
#pragma unroll
      for (int tn = 0; tn < kTN; ++tn) a.c[tm][tn] = acc4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  __device__ __forceinline__ float reduce_over_cols(float v) const {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  }
  __device__ __forceinline__ bool col_leader() const { return (lane & 15) == 0; }

  // This thread's four 16-byte pieces of one operand's K stage.  K-contiguous: rows
  // t/8 + 32*j, K values 4*(t%8) .. +4.  K-major: K rows 4*(t/32) + j, columns 4*(t%32) .. +4.
  // Rows / columns past the matrix are clamped (their results are discarded), pieces past
  // k_end are zero (a K-contiguous piece that straddles it is loaded whole: its row is
  // padded to it, and the other operand is zero there).
  template <bool kKMajor>
  static __device__ __forceinline__ void load(const Operand<float>& x, int k0, int k_end,
                                              acc4_t (&r)[4]) {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = kKMajor ? k0 + 4 * (t >> 5) + j : k0 + 4 * (t & 7);
      const int64_t at =
          kKMajor ? (int64_t)k * x.ld + min(x.row0 + 4 * (t & 31), x.rows - 4)
                  : (int64_t)min(x.row0 + (t >> 3) + 32 * j, x.rows - 1) * x.ld + k;
      r[j] = k < k_end ? *reinterpret_cast<const acc4_t*>(x.ptr + at)
                       : acc4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  template <bool kKMajor>
  static __device__ __forceinline__ void store(char* op_stage, const acc4_t (&r)[4]) {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = kKMajor ? 4 * (t & 31) + j : (t >> 3) + 32 * j;
      const int chunk = kKMajor ? t >> 5 : t & 7;
      const acc4_t v = kKMajor ? acc4_t{r[0][j], r[1][j], r[2][j], r[3][j]} : r[j];
      *reinterpret_cast<acc4_t*>(op_stage + row * 128 + ((chunk ^ ((row >> 1) & 7)) * 16)) = v;
    }
  }

  template <bool kAKMajor, bool kBKMajor>
  __device__ __forceinline__ void mainloop_ex(const Operand<float>& A, const Operand<float>& B,
                                              int k_begin, int k_end, Acc& acc,
                                              char* smem) const {
    zero(acc);
    acc4_t ra[4], rb[4];
    const int slot = (lane >> 4) ^ ((lane >> 1) & 7);
    const char* a_base = smem + (wm * 64 + (lane & 15)) * 128;
    const char* b_base = smem + kOperandBytes + (wn * 64 + (lane & 15)) * 128;
    load<kAKMajor>(A, k_begin, k_end, ra);
    load<kBKMajor>(B, k_begin, k_end, rb);
    store<kAKMajor>(smem, ra);
    store<kBKMajor>(smem + kOperandBytes, rb);
    __syncthreads();
    int cur = 0;
    for (int k0 = k_begin; k0 < k_end; k0 += kBK, cur ^= 1) {
      const bool more = k0 + kBK < k_end;
      if (more) {
        load<kAKMajor>(A, k0 + kBK, k_end, ra);
        load<kBKMajor>(B, k0 + kBK, k_end, rb);
      }
      const int stage = cur * kStageBytes;
#pragma unroll
      for (int kg = 0; kg < 2; ++kg) {
        const int at = stage + ((slot ^ (kg * 4)) * 16);
        acc4_t fa[kTM], fb[kTN];
#pragma unroll
        for (int tm = 0; tm < kTM; ++tm)
          fa[tm] = *reinterpret_cast<const acc4_t*>(a_base + at + tm * 16 * 128);
#pragma unroll
        for (int tn = 0; tn < kTN; ++tn)
          fb[tn] = *reinterpret_cast<const acc4_t*>(b_base + at + tn * 16 * 128);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int tm = 0; tm < kTM; ++tm)
#pragma unroll
            for (int tn = 0; tn < kTN; ++tn)
              acc.c[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[tm][j], fb[tn][j],
                                                                   acc.c[tm][tn], 0, 0, 0);
      }
      if (more) {
        char* next = smem + (cur ^ 1) * kStageBytes;
        store<kAKMajor>(next, ra);
        store<kBKMajor>(next + kOperandBytes, rb);
      }
      __syncthreads();
    }
  }

  __device__ __forceinline__ void mainloop_set(const float* __restrict__ A, int64_t lda,
                                               int a_row0, int a_rows,
                                               const float* __restrict__ B, int64_t ldb,
                                               int b_row0, int b_rows, int k_begin, int k_end,
                                               Acc& acc, char* smem) const {
    const Operand<float> a = {A, lda, a_row0, a_rows};
    const Operand<float> b = {B, ldb, b_row0, b_rows};
    mainloop_ex<false, false>(a, b, k_begin, k_end, acc, smem);
  }
};

}  // namespace tlce
