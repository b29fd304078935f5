// 256x256 bf16/f16 MFMA tile engines for gfx950 (CDNA4), wave64.
//
// Both compute C[i][j] = sum_k A[i][k] * B[j][k] for one 256x256 tile.  The
// register-staged engine (any K that is a multiple of 8, operands K-contiguous,
// row-major [rows, K]): 512 threads = 8 waves in a 2 (A rows) x 4 (B rows) grid; each
// wave owns a 128x64 sub-tile as 4x2 v_mfma_f32_32x32x16 blocks (128 fp32
// accumulator registers per lane), two waves per SIMD.
//
// LDS: two stages of (A 256x64 + B 256x64) 2-byte elements = 2 x 64 KiB of the
// CU's 160 KiB.  A tile row is 128 bytes = eight 16-byte chunks; chunk c of
// row r lives at chunk slot c ^ ((r >> 1) & 7), which makes both the 16-byte
// staging writes and the 16-byte MFMA fragment reads hit all 64 banks.
//
// Accumulator layout of one 32x32 block (lane l, register q of 16):
//   row = 8*(q/4) + 4*(l/32) + q%4,   col = l%32.
// A/B fragment of one block for K-slice ks: lane l supplies row l%32,
// K = 16*ks + 8*(l/32) .. +8  (one 16-byte chunk).
#pragma once

#include <type_traits>

#include "tlce_common.h"

namespace tlce {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

template <typename T> struct MfmaOp;
template <> struct MfmaOp<__bf16> {
  using V8 = bf16x8_t;
  static __device__ __forceinline__ f32x16_t mma(V8 a, V8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct MfmaOp<_Float16> {
  using V8 = f16x8_t;
  static __device__ __forceinline__ f32x16_t mma(V8 a, V8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// Its thread <-> tile-element mapping.
template <typename T_>
struct MfmaTileLayout {
  using T = T_;
  using Op = MfmaOp<T>;
  using V8 = typename Op::V8;

  static constexpr int kTile = 256;     // BM == BN
  static constexpr int kTileB = kTile;
  static constexpr int kWavesN = 4;     // waves along B rows
  static constexpr int kThreads = 2 * kWavesN * 64;
  static constexpr int kTM = 4;         // 32-row blocks per wave along A rows
  static constexpr int kTN = 2;         // 32-col blocks per wave along B rows
  static constexpr int kCols = kTN;          // tile columns owned per thread
  static constexpr int kRows = kTM * 16;     // tile rows held per owned column
  static constexpr int kShare = 4;           // threads that hold the same column
  static constexpr int kPlanes = 1;
  static constexpr int kWavesPerSimd = 1;
  static constexpr bool kPrecise = false;    // hardware exp / rcp approximations in the epilogues
  static constexpr bool kReadsWhereUsed = false;
  static_assert(kWavesN * kTN * 32 == kTile, "waves must tile the 256 B rows");

  struct Acc { f32x16_t c[kTM][kTN]; };

  int lane, wave, wm, wn;

  __device__ __forceinline__ MfmaTileLayout() {
    lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    wm = wave / kWavesN;
    wn = wave % kWavesN;
  }

  // An empty asm that "modifies" the lane index: values derived from it before
  // this point are not reused after it, so a kernel that loops over tiles can
  // keep the compiler from hoisting (and then spilling) per-lane addresses.
  __device__ __forceinline__ void forget_lane_invariants() { asm volatile("" : "+v"(lane)); }

  __device__ __forceinline__ int col(int j) const {
    return wn * (kTN * 32) + j * 32 + (lane & 31);
  }
  __device__ __forceinline__ int row(int i) const {
    return wm * 128 + (i >> 4) * 32 + ((i >> 2) & 3) * 8 + (lane >> 5) * 4 + (i & 3);
  }
  __device__ __forceinline__ int share_slot() const { return wm * 2 + (lane >> 5); }
  static __device__ __forceinline__ float get(const Acc& a, int j, int i) {
    return a.c[i >> 4][j][i & 15];
  }
  static __device__ __forceinline__ void set(Acc& a, int j, int i, float v) {
    a.c[i >> 4][j][i & 15] = v;
  }
  static __device__ __forceinline__ void zero(Acc& a) {
#pragma unroll
    for (int tm = 0; tm < kTM; ++tm)
#pragma unroll
      for (int tn = 0; tn < kTN; ++tn)
#pragma unroll
        for (int q = 0; q < 16; ++q) a.c[tm][tn][q] = 0.0f;
  }
  // Sum over the lanes that hold the same tile row (the 32 lanes of a half-wave).
  __device__ __forceinline__ float reduce_over_cols(float v) const {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  }
  __device__ __forceinline__ bool col_leader() const { return (lane & 31) == 0; }
};

// Register-staged engine: global -> VGPR -> LDS, two 64-wide K stages.  Takes
// any K that is a multiple of 8 (zero-fills the tail); used when the hidden
// size is not a multiple of 32.
template <typename T_>
struct MfmaEngine : MfmaTileLayout<T_> {
  using Base = MfmaTileLayout<T_>;
  using T = T_;
  using Op = typename Base::Op;
  using V8 = typename Base::V8;
  using Acc = typename Base::Acc;
  using Base::kTile;
  using Base::kTM;
  using Base::kTN;
  using Base::lane;
  using Base::wm;
  using Base::wn;
  static constexpr int kBK = 64;
  static constexpr int kRowBytes = kBK * 2;                  // 128
  static constexpr int kStageBytes = 2 * kTile * kRowBytes;  // 65536
  static constexpr int kSmemBytes = 2 * kStageBytes;         // 131072
  static constexpr bool kHasKMajor = false;

  // acc += A[a_row0 .. +256, k_begin .. k_end) * B[b_row0 .. +256, same K)^T.
  // Rows past a_rows / b_rows are clamped to the last valid row (their results
  // are discarded by the caller); K past k_end is zero-filled.  k_begin and
  // k_end are multiples of 8 and lda/ldb multiples of 8 (16-byte chunks).
  __device__ __forceinline__ void mainloop(const T* __restrict__ A, int64_t lda, int a_row0,
                                           int a_rows, const T* __restrict__ B, int64_t ldb,
                                           int b_row0, int b_rows, int k_begin, int k_end,
                                           Acc& acc, char* smem) const {
    const int tid = threadIdx.x;
    const int c = tid & 7;
    const int r0 = tid >> 3;
    const int pc = c ^ ((tid >> 4) & 7);

    const T* ap[4];
    const T* bp[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int ar = min(a_row0 + r0 + 64 * j, a_rows - 1);
      const int br = min(b_row0 + r0 + 64 * j, b_rows - 1);
      ap[j] = A + (int64_t)ar * lda + k_begin + c * 8;
      bp[j] = B + (int64_t)br * ldb + k_begin + c * 8;
    }
    const int st_off = r0 * kRowBytes + pc * 16;

    const int swz = (lane >> 1) & 7;
    const int hi = lane >> 5;
    const int a_frag = (wm * 128 + (lane & 31)) * kRowBytes;
    const int b_frag = kTile * kRowBytes + (wn * 64 + (lane & 31)) * kRowBytes;

    uint4 ra[4], rb[4];

    // A chunk past k_end re-reads the row's first chunk (always in bounds) and
    // is zeroed in registers, so the loads stay unconditional global loads.
    auto gload = [&](int k0) {
      const bool ok = (k0 + c * 8) < k_end;
      const int64_t back = ok ? 0 : (int64_t)(k0 - k_begin + c * 8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ra[j] = *reinterpret_cast<const uint4*>(ap[j] - back);
        rb[j] = *reinterpret_cast<const uint4*>(bp[j] - back);
        if (!ok) {
          ra[j] = make_uint4(0u, 0u, 0u, 0u);
          rb[j] = make_uint4(0u, 0u, 0u, 0u);
        }
        ap[j] += kBK;
        bp[j] += kBK;
      }
    };
    auto sstore = [&](int stage) {
      char* base = smem + stage * kStageBytes + st_off;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<uint4*>(base + j * 64 * kRowBytes) = ra[j];
        *reinterpret_cast<uint4*>(base + kTile * kRowBytes + j * 64 * kRowBytes) = rb[j];
      }
    };
    auto compute = [&](int stage) {
      const char* base = smem + stage * kStageBytes;
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        const int slot = ((2 * ks + hi) ^ swz) * 16;
        V8 af[kTM], bf[kTN];
#pragma unroll
        for (int tm = 0; tm < kTM; ++tm)
          af[tm] = __builtin_bit_cast(
              V8, *reinterpret_cast<const uint4*>(base + a_frag + tm * 32 * kRowBytes + slot));
#pragma unroll
        for (int tn = 0; tn < kTN; ++tn)
          bf[tn] = __builtin_bit_cast(
              V8, *reinterpret_cast<const uint4*>(base + b_frag + tn * 32 * kRowBytes + slot));
#pragma unroll
        for (int tm = 0; tm < kTM; ++tm)
#pragma unroll
          for (int tn = 0; tn < kTN; ++tn) acc.c[tm][tn] = Op::mma(af[tm], bf[tn], acc.c[tm][tn]);
      }
    };

    const int nk = (k_end - k_begin + kBK - 1) / kBK;
    gload(k_begin);
    sstore(0);
    __syncthreads();
    for (int it = 0; it < nk; ++it) {
      const int cur = it & 1;
      const bool more = (it + 1) < nk;
      if (more) gload(k_begin + (it + 1) * kBK);
      compute(cur);
      if (more) sstore(cur ^ 1);
      __syncthreads();
    }
  }

  // acc = A * B^T (same operands as mainloop).
  __device__ __forceinline__ void mainloop_set(const T* __restrict__ A, int64_t lda, int a_row0,
                                               int a_rows, const T* __restrict__ B, int64_t ldb,
                                               int b_row0, int b_rows, int k_begin, int k_end,
                                               Acc& acc, char* smem) const {
    Base::zero(acc);
    mainloop(A, lda, a_row0, a_rows, B, ldb, b_row0, b_rows, k_begin, k_end, acc, smem);
  }
};

// Thread <-> tile-element mapping of the direct-to-LDS engine: 4 waves (2 along the A
// rows x 2 along the B rows), each 128x128 as 8x8 v_mfma_f32_16x16x32 blocks.
//
// Why 16x16x32 and not 32x32x16, whose operand registers are read half as often: with
// real operand values the matrix pipes run at the part's power limit, and per FLOP the
// 16x16x32 instruction moves its accumulator half as often (K = 32 per accumulation).
// Measured on registers alone with normally distributed bf16 operands: 2050 against
// 1780 TFLOP/s (2440 / 2480 with all-zero operands).  That holds only while the A
// operand stays the same over a run of MFMAs (a change of A stalls the next issue by
// about 5 cycles: 1820 TFLOP/s on zeros when A changes every time), hence 8 columns of
// B per A fragment.
//
// Accumulator layout of one 16x16 block (lane l, register q of 4):
//   row = 4*(l/16) + q,   col = l%16.
// A/B fragment of one block for a 32-wide K slice: lane l supplies row l%16,
// K = 8*(l/16) .. +8  (one 16-byte chunk).
typedef float acc4_t __attribute__((ext_vector_type(4)));

template <typename T_, int kTN_ = 8>
struct DirectTileLayout {
  using T = T_;
  static constexpr int kTile = 256;
  static constexpr int kThreads = 256;
  static constexpr int kTM = 8;                  // 16-row blocks per wave along A rows
  static constexpr int kTN = kTN_;               // 16-row blocks per wave along B rows
  static constexpr int kTileB = 32 * kTN;        // the tile's B rows (256, or fewer: narrow tiles)
  static constexpr int kWaveB = 16 * kTN;        // B rows of a wave
  static constexpr int kCols = kTN;              // tile columns owned per thread
  static constexpr int kRows = kTM * 4;          // tile rows held per owned column
  static constexpr int kShare = 8;               // threads that hold the same column
  static constexpr int kStageCols = 2;           // owned columns per quarter of the tile
  static constexpr int kWavesPerSimd = 1;
  static constexpr bool kPrecise = false;
  static constexpr bool kReadsWhereUsed = kTN == 8;   // read() in place of get()

  struct Acc { acc4_t c[kTM][kTN]; };

  int lane, wave, wm, wn;

  __device__ __forceinline__ DirectTileLayout() {
    lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    wm = wave >> 1;
    wn = wave & 1;
  }
  __device__ __forceinline__ void forget_lane_invariants() { asm volatile("" : "+v"(lane)); }
  __device__ __forceinline__ int col(int j) const { return wn * kWaveB + j * 16 + (lane & 15); }
  // The tile columns that have owned index j in some thread: number t of them.
  static constexpr int kTokensPerIndex = 32;
  static __device__ __forceinline__ int token_of_index(int j, int t) {
    return (t >> 4) * kWaveB + j * 16 + (t & 15);
  }
  // Position of this lane's column among those with the same owned index.
  __device__ __forceinline__ int position_in_index() const { return wn * 16 + (lane & 15); }
  __device__ __forceinline__ int row(int i) const {
    return wm * 128 + (i >> 2) * 16 + (lane >> 4) * 4 + (i & 3);
  }
  __device__ __forceinline__ int share_slot() const { return wm * 4 + (lane >> 4); }
  static __device__ __forceinline__ float get(const Acc& a, int j, int i) {
    return a.c[i >> 2][j][i & 3];
  }
  // The same, copied to a VGPR at this place: left to itself the compiler copies all 256
  // accumulators at once where the first is used.
  static __device__ __forceinline__ float read(const Acc& a, int j, int i) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a.c[i >> 2][j][i & 3]));
    return v;
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
  // Sum over the lanes that hold the same tile row (a group of 16 lanes).
  __device__ __forceinline__ float reduce_over_cols(float v) const {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  }
  __device__ __forceinline__ bool col_leader() const { return (lane & 15) == 0; }
};

// Four-wave direct-to-LDS engine (K multiple of 64): 256 threads, each wave a
// 128x128 sub-tile (256 accumulator registers, one wave per SIMD).  Operands go
// global -> LDS with global_load_lds_dwordx4 (no VGPR staging, no ds_write) into two
// 64-wide K stages of 64 KiB; every wave load instruction moves 1 KiB made of full
// 128-byte (or 512-byte) row segments.
//
// Either operand can be stored in one of two ways:
//   K-contiguous  X[row][k]  (the projection's hidden and weight rows, the
//                 logit-gradient panel as seen by grad_hidden);
//   K-major       X[k][row]  (weight as seen by grad_hidden, hidden and the
//                 logit-gradient panel as seen by grad_weight), read from LDS
//                 with the transposing ds_read_b64_tr_b16, so no transposed
//                 copy of any matrix is ever made in HBM.
//
// LDS layouts of one operand stage (32 KiB):
//   K-contiguous: 256 rows x 128 B; 16-byte chunk c of row r in slot
//                 c ^ ((r >> 1) & 7): any 16 consecutive rows of one chunk cover
//                 all 64 banks.
//   K-major:      64 K rows x 512 B; 16-byte chunk c of K row k in slot
//                 c ^ (4 * (k & 3)) ^ (2 * ((k >> 3) & 1)): the eight K rows (0..3 and
//                 8..11) x 32 bytes that half a wave reads at once fall into eight
//                 different eighths of the banks.
// ds_read_b64_tr_b16 works on groups of 16 lanes: lane i of a group addresses
// 4 consecutive elements, and lane l receives element l%4 of the chunks of
// lanes l/4, 4 + l/4, 8 + l/4, 12 + l/4.  With lane i addressing K row i/4,
// columns 4*(i%4).. of a 4 x 16 block, lane l ends up with 4 consecutive K
// values of column l: half an MFMA fragment.
//
// A K range that ends inside a 64-row slab of a K-major operand (a vocabulary or row
// count that is no multiple of 64) takes its last tile from a zero-padded copy of those
// rows: the scalar base of the last tile is another pointer, nothing else changes.
// Before, such vocabularies went through transposed copies of the head and of the
// logit-gradient panel and four contractions.
//
// Loads use the scalar-base form: tile base and K position live in SGPRs, the
// per-lane byte offsets (row clamp and slot swizzle folded in) are computed
// once per tile, so a load costs three scalar instructions and no VALU work.
//
// Software pipeline of one wave (the only wave on its SIMD; it issues in
// order and an MFMA occupies its pipe for 16 cycles): one K step = 2 slices of 32 =
// 2 x 8 groups of 8 MFMAs (A block q, B blocks 0..7).  After every MFMA at most one
// fragment read or load instruction follows.
//   reads : B fragments are held twice (all eight are needed by every group), those of
//           the next slice are read in the first groups of the current one; an A
//           fragment is needed by one group only, so its registers are refilled for
//           the next slice right after that group.  The barrier that makes the next
//           tile visible sits before group 2 of slice 1, when the last fragment of the
//           current stage (A block 7, read in group 0) has arrived.
//   loads : of the next tile's 16, kLoadsAfterBarrier go out in the groups right after
//           the barrier of the previous step, the others in the first groups of the
//           step, two per group: bunched four to a group the kernels lose 2 to 4 %, all
//           16 right after the barrier 4 %, 6 there and 10 in the step 8 %.
//   touches: the workgroups of an XCD share their operand strips through its L2, but all
//           of them wait for whichever fetch misses it, and one tile of lead (about
//           1 us) does not cover a fetch from beyond L2.  Once per step each wave reads
//           one dword from 64 of the K tile's 128-byte lines, kTouchAhead tiles ahead,
//           into a scrap of LDS nobody reads: neighbouring workgroups (even and odd tile
//           index along the other operand) take the two halves of a strip, so between
//           them the whole tile is in L2 before its loads are issued.
//
// Measured on one block of 8192 rows, H = 4096, V = 151936 (ms per contraction,
// 32x32x16 engine -> 16x16x32 with the accumulators in AGPRs -> with touches):
// exponentiated logits 8.1 -> 7.65 -> 7.3, grad_hidden 7.75 -> 7.25 -> 6.95, grad_weight
// 7.85 -> 7.3 -> 7.25, forward statistics 7.8 -> 7.5 -> 7.2 (1.38 to 1.47 PFLOP/s;
// grad_hidden's pipes are busy 0.835 of the cycles at 1.65 GHz, i.e. at the power
// limit).  With no loads in the K loop grad_hidden takes 5.4 ms, with every load an L2
// hit 6.2: what is left is the energy of moving operands.
template <typename T>
struct Operand {
  const T* ptr;   // matrix base
  int64_t ld;     // elements between consecutive stored rows
  int row0;       // first tile row (K-contiguous) or first tile column (K-major)
  int rows;       // valid rows / columns of the matrix; accesses beyond are clamped
  // K-major: K rows from k_full on (a multiple of 64; the matrix has fewer than 64 more)
  // are read from `tail`, a [64, ld] copy of them with zero rows after the last.
  // K-contiguous first operand of the engine that has column tails: the columns after the
  // last whole 64 are read from `tail`, a [rows, 64] copy with zero columns after the last.
  const T* tail = nullptr;
  int k_full = 0x7fffffff;
};

template <typename T> struct DirectMfma;
// The MFMAs are written as asm so that the accumulators stay in the AGPR file: left to
// the builtin, the allocator moves some of the 64 blocks through VGPRs inside the loop
// (44 to 116 copies, each behind a full MFMA latency, per K step).  The waits for the
// LDS reads that fill a and b are the compiler's, which tracks asm operands; what it
// does not know is the result latency, so mainloop_ex ends on mfma_drain().
template <> struct DirectMfma<__bf16> {
  static __device__ __forceinline__ void mma(bf16x8_t a, bf16x8_t b, acc4_t& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mma_set(bf16x8_t a, bf16x8_t b, acc4_t& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ acc4_t mma_builtin(bf16x8_t a, bf16x8_t b, acc4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct DirectMfma<_Float16> {
  static __device__ __forceinline__ void mma(f16x8_t a, f16x8_t b, acc4_t& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mma_set(f16x8_t a, f16x8_t b, acc4_t& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ acc4_t mma_builtin(f16x8_t a, f16x8_t b, acc4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <typename T_, int kPlanes_, bool kColumnTail = false, int kTN_ = 8>
struct DirectToLdsEngine : DirectTileLayout<T_, kTN_> {
  using Base = DirectTileLayout<T_, kTN_>;
  using T = T_;
  // The K loop's passes over the planes of the operands (kPlanes == 1: one over the
  // matrices themselves).  Plane of A and of B in pass s: nibble s of these.
  static constexpr int kPlanes = kPlanes_;
  static constexpr int kPasses = kPlanes == 1 ? 1 : 6;
  static constexpr unsigned kPassPlaneA = kPlanes == 1 ? 0u : 0x001102u;
  static constexpr unsigned kPassPlaneB = kPlanes == 1 ? 0u : 0x010120u;
  static_assert(kPlanes == 1 || kPlanes == 3, "matrices as they are, or float32 in three planes");
  static_assert(!kColumnTail || kPlanes == 1, "planes are padded to whole K tiles");
  static constexpr bool kPrecise = kPlanes > 1;              // float32 in, float32 epilogues
  using Op = DirectMfma<T_>;
  using V8 = typename MfmaOp<T_>::V8;
  using Acc = typename Base::Acc;
  using Base::kTile;
  using Base::kTM;
  using Base::kTN;
  using Base::lane;
  using Base::wave;
  using Base::wm;
  using Base::wn;
  static constexpr int kBK = 64;
  static constexpr int kOperandBytes = kTile * kBK * 2;      // 32768
  static constexpr int kStageBytes = 2 * kOperandBytes;      // 65536
  static constexpr int kTouchBytes = 4 * 256;                // where the L2 touches land
  static constexpr bool kNarrow = kTN_ < 8;
  static constexpr int kNarrowStages = 3;
  static constexpr int kNarrowStageBytes = (kTile + Base::kTileB) * kBK * 2;
  static constexpr int kSmemBytes =
      kNarrow ? kNarrowStages * kNarrowStageBytes : 2 * kStageBytes + kTouchBytes;
  static_assert(!kNarrow || (kPlanes == 1 && !kColumnTail), "narrow tiles: matrices as they are");
  static constexpr int kLoads = 8;                           // per wave, operand and K tile
  static constexpr int kLoadsB = kNarrow ? kTN_ : kLoads;    // of a K-contiguous second operand
  static constexpr int kTouchAhead = 2;                      // K tiles
  static constexpr int kLoadsAfterBarrier = 12;              // of the 16 of both operands
  static constexpr bool kHasKMajor = true;

  typedef short v4s_t __attribute__((ext_vector_type(4)));
  typedef short v8s_t __attribute__((ext_vector_type(8)));

  static __device__ __forceinline__ void load_to_lds(unsigned lds_addr, unsigned byte_offset,
                                                     const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr), "v"(byte_offset), "s"(base)
                 : "memory", "m0");
  }

  static __device__ __forceinline__ void touch(unsigned lds_addr, unsigned byte_offset,
                                               const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds_addr), "v"(byte_offset), "s"(base)
                 : "memory", "m0");
  }

  static __device__ __forceinline__ int64_t readfirstlane64(int64_t x) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)x);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(x >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
  }

  // Per-lane byte offset of cache line `line` (0..255, 128 bytes each) of an operand's K tile.
  template <bool kKMajor>
  static __device__ __forceinline__ unsigned line_offset(const Operand<T>& x, int line) {
    if (!kKMajor) {
      return (unsigned)((int64_t)(min(x.row0 + line, x.rows - 1) - x.row0) * x.ld * kPlanes * 2);
    } else {
      const int last_chunk = x.rows / 8 - 1 - x.row0 / 8;
      return (unsigned)((int64_t)(line >> 2) * x.ld * kPlanes * 2 +
                        min((line & 3) * 8, last_chunk) * 16);
    }
  }

  // Loader state of one operand: where this wave's eight 1 KiB pieces of a K
  // tile come from and where they land.
  struct Loader {
    unsigned off[kLoads];   // per-lane byte offsets from the K tile's base
    unsigned fill;          // LDS address of this wave's first piece in stage 0
    const char* next;       // base address of the next K tile to request
    int64_t step;           // bytes between consecutive K tiles
    const char* last;       // K-major: base address of the last K tile (the operand's tail
                            // when the K range ends inside a 64-row slab); column tails:
                            // the tail's first row of this tile
    unsigned last_off[kColumnTail ? kLoads : 1];   // column tails: `off` of the last K tile
    const char* begin;      // base address of the first K tile in plane 0
    int64_t plane;          // bytes from one plane to the next
  };

  template <bool kKMajor, bool kTail = false, int kN = kLoads>
  __device__ __forceinline__ Loader make_loader(const Operand<T>& x, int k_begin, int nk,
                                                unsigned lds_op) const {
    Loader ld;
    if (!kKMajor) {
      // this wave fills tile rows [64w, 64w+64) (of kN loads: [8 kN w, ...)), eight rows per
      // instruction
#pragma unroll
      for (int j = 0; j < kN; ++j) {
        const int r = wave * (8 * kN) + j * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        const int rr = min(x.row0 + r, x.rows - 1) - x.row0;
        ld.off[j] = (unsigned)((int64_t)rr * x.ld * kPlanes * 2 + chunk * 16);
      }
      ld.fill = __builtin_amdgcn_readfirstlane(lds_op + (unsigned)(wave * 8 * kN * 128));
      ld.next = reinterpret_cast<const char*>(x.ptr + (int64_t)x.row0 * x.ld * kPlanes + k_begin);
      ld.step = kBK * 2;
      ld.last = nullptr;
      if constexpr (kTail) {
        ld.last = reinterpret_cast<const char*>(x.tail + (int64_t)x.row0 * kBK);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
          const int r = wave * 64 + j * 8 + (lane >> 3);
          const int chunk = (lane & 7) ^ ((r >> 1) & 7);
          ld.last_off[j] = (unsigned)((min(x.row0 + r, x.rows - 1) - x.row0) * kBK * 2 + chunk * 16);
        }
      }
    } else {
      // this wave fills K rows [16w, 16w+16) of the slab, two rows per instruction
      const int last_chunk = x.rows / 8 - 1 - x.row0 / 8;   // relative to the tile
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int kr = wave * 16 + j * 2 + (lane >> 5);
        const int swz = (4 * (kr & 3)) ^ (2 * ((kr >> 3) & 1));
        const int chunk = min((lane & 31) ^ swz, last_chunk);
        ld.off[j] = (unsigned)((int64_t)kr * x.ld * kPlanes * 2 + chunk * 16);
      }
      ld.fill = __builtin_amdgcn_readfirstlane(lds_op + (unsigned)(wave * 16 * 512));
      const int k_last = k_begin + (nk - 1) * kBK;
      ld.last = reinterpret_cast<const char*>(
          (k_last >= x.k_full ? x.tail : x.ptr + (int64_t)k_last * x.ld) + x.row0);
      ld.next = kPlanes == 1 && nk == 1
                    ? ld.last
                    : reinterpret_cast<const char*>(x.ptr + (int64_t)k_begin * x.ld * kPlanes +
                                                    x.row0);
      ld.step = (int64_t)kBK * x.ld * kPlanes * 2;
    }
    ld.begin = ld.next;
    ld.plane = x.ld * 2;
    return ld;
  }

  // Fragment addressing of one operand for this lane: LDS byte offset within the
  // operand stage of block 0, K slice 0.
  template <bool kKMajor, int kWaveRows = 128>
  __device__ __forceinline__ int reader_base(int wave_block) const {
    if (!kKMajor) {
      return (wave_block * kWaveRows + (lane & 15)) * 128 +
             (((lane >> 4) ^ ((lane >> 1) & 7)) * 16);
    } else {
      const int g = lane >> 4;           // 16-lane group
      const int i = lane & 15;
      const int kr = 8 * g + (i >> 2);   // K row within the 32-wide slice, first half
      const int swz = (4 * (i >> 2)) ^ (2 * (g & 1));
      const int chunk = wave_block * 16 + ((i & 3) >> 1);
      return kr * 512 + (chunk ^ swz) * 16 + (i & 1) * 8;
    }
  }

  template <bool kKMajor>
  __device__ __forceinline__ V8 read_frag(const char* op_stage, int base, int ks, int b) const {
    if (!kKMajor) {
      // slice 1 is chunks 4..7: the slot's bit 2 flips; block b starts 16 rows further
      return __builtin_bit_cast(
          V8, *reinterpret_cast<const uint4*>(op_stage + ((base ^ (ks * 64)) + b * 16 * 128)));
    } else {
      typedef __attribute__((address_space(3))) v4s_t* lds_v4s_ptr;
      // block b is chunks 2b, 2b + 1 of the wave's 16: address bits 5..7
      const char* p0 = op_stage + (base ^ (b * 32)) + ks * 32 * 512;
      const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_v4s_ptr)(uintptr_t)(unsigned)(uintptr_t)p0);
      const v4s_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_v4s_ptr)(uintptr_t)(unsigned)(uintptr_t)(p0 + 4 * 512));
      v8s_t v;
      v[0] = lo[0]; v[1] = lo[1]; v[2] = lo[2]; v[3] = lo[3];
      v[4] = hi4[0]; v[5] = hi4[1]; v[6] = hi4[2]; v[7] = hi4[3];
      return __builtin_bit_cast(V8, v);
    }
  }

  // Waits until the last MFMAs' results can be read (19 cycles for 16x16 blocks); takes
  // the accumulators written last so that no read of them is moved above it.
  static __device__ __forceinline__ void mfma_drain(Acc& acc) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 7"
                 : "+a"(acc.c[7][0]), "+a"(acc.c[7][1]), "+a"(acc.c[7][2]), "+a"(acc.c[7][3]),
                   "+a"(acc.c[7][4]), "+a"(acc.c[7][5]), "+a"(acc.c[7][6]), "+a"(acc.c[7][7]));
    __builtin_amdgcn_sched_barrier(0);
  }

  // Every accumulator as a value of its own, in its register, at this place.
  static __device__ __forceinline__ void pin(Acc& acc) {
#pragma unroll
    for (int q = 0; q < kTM; ++q)
#pragma unroll
      for (int t = 0; t < kTN; ++t) asm volatile("" : "+a"(acc.c[q][t]));
  }

  // acc = A-tile * B-tile^T over K in [k_begin, k_end), not empty and a multiple of 64 wide
  // (with column tails, of K-contiguous operands: 65 wide at least and no such multiple, and
  // the rows of B hold zeros up to the next one)
  // (the first 64 MFMAs take a zero constant as their addend, which saves zeroing 256
  // accumulator registers per tile).
  // K-contiguous operand: tile rows row0 .. row0+256 of x (rows clamped to
  // x.rows - 1).  K-major operand: tile columns row0 .. row0+256 of x (16-byte
  // column chunks clamped to the last valid one; x.rows is a multiple of 8); the K
  // rows in [k_begin, k_end) must exist up to k_full, and in the tail from there on.
  template <bool kAKMajor, bool kBKMajor>
  __device__ __forceinline__ void mainloop_ex(const Operand<T>& A, const Operand<T>& B,
                                              int k_begin, int k_end, Acc& acc,
                                              char* smem) const {
    if constexpr (kNarrow) {
      static_assert(!kBKMajor, "narrow tiles: a K-contiguous second operand");
      narrow_loop<kAKMajor>(A, B, k_begin, k_end, acc, smem);
    } else {
      wide_loop<kAKMajor, kBKMajor>(A, B, k_begin, k_end, acc, smem);
    }
  }

  // Narrow tiles: 64 or 128 rows of B.  The last token tile of a call holds what is left over
  // 256, and a short call holds nothing else: 64 rows in a tile of 256 do four times the
  // operations.  A K tile is short here (32 or 64 MFMAs a wave), so what bounds it is the
  // operands' way: three stages, of which two are on the way while one is contracted, and the
  // fragments of the next slice are read between the MFMAs of this one.  The sums are the wide
  // loop's, in its order.  The MFMAs are the builtin's: few accumulators stay where they are
  // without help, and the compiler sees to their hazards.  Without the reads in between (left to
  // the compiler: two fragments, a wait, eight MFMAs) a tile took as long as a wide one.
  // 64 rows, H = 1024, V = 32000: exponentiated logits 29 -> 16 us, grad_hidden 24 -> 16; a step of
  // 64 rows over H = 4096, V = 151936 1050 -> 919 us (of 128 rows 1130 -> 1009), where its bytes
  // take 790.  After whole tiles less is gained, as the neighbours share the head's strips: 1036
  // rows of the small head 91 -> 85 us of exponentiated logits, 1610 rows over V = 151936 1646 ->
  // 1605, 8212 rows over H = 1024, V = 65536 2.90 -> 2.84 ms a step.
  template <bool kAKMajor>
  __device__ __forceinline__ void narrow_loop(const Operand<T>& A, const Operand<T>& B,
                                              int k_begin, int k_end, Acc& acc,
                                              char* smem) const {
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    const int nk = (k_end - k_begin) / kBK;
    Loader la = make_loader<kAKMajor>(A, k_begin, nk, lds0);
    Loader lb = make_loader<false, false, kLoadsB>(B, k_begin, nk, lds0 + kOperandBytes);
    const int ra = reader_base<kAKMajor>(wm);
    const int rb = reader_base<false, Base::kWaveB>(wn);
    auto advance = [&](int k) {
      la.next = kAKMajor && k == nk - 1 ? la.last : la.next + la.step;
      lb.next += lb.step;
    };
    // load number q of the K tile the loaders stand at
    constexpr int kTileLoads = kLoads + kLoadsB;
    auto issue_one = [&](unsigned s_off, int q) {
      if (q < kLoads) load_to_lds(la.fill + s_off + q * 1024, la.off[q], la.next);
      else load_to_lds(lb.fill + s_off + (q - kLoads) * 1024, lb.off[q - kLoads], lb.next);
    };
    auto issue = [&](int stage) {
#pragma unroll
      for (int q = 0; q < kTileLoads; ++q) issue_one((unsigned)(stage * kNarrowStageBytes), q);
    };
    // fragment number r of a slice: those of B, which every group needs, first
    constexpr int kFrags = kTN + kTM;
    V8 fa[2][kTM], fb[2][kTN];
    auto read_one = [&](const char* stage, int s, int r) {
      if (r < kTN) fb[s][r] = read_frag<false>(stage + kOperandBytes, rb, s, r);
      else fa[s][r - kTN] = read_frag<kAKMajor>(stage, ra, s, r - kTN);
    };
    unsigned cur = 0;   // LDS offset of the current K tile's stage
    // left: how many K tiles follow (0, 1, 2, or 3 for "three or more")
    auto step = [&](int k, auto left_tag) {
      constexpr int kLeft = decltype(left_tag)::value;
      const unsigned nxt = cur == 2 * kNarrowStageBytes ? 0 : cur + kNarrowStageBytes;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (s == 1 && kLeft >= 1) {
          // K tile k + 1 is complete and visible from here on, and the current stage free
          asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kLeft >= 2 ? kTileLoads : 0) : "memory");
          __syncthreads();
          if (kLeft >= 3) advance(k + 3);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < kTM; ++q) {
#pragma unroll
          for (int t = 0; t < kTN; ++t)
            acc.c[q][t] = Op::mma_builtin(fa[s][q], fb[s][t], acc.c[q][t]);
#pragma unroll
          for (int r = 2 * q; r < 2 * q + 2; ++r) {
            if (r < kFrags && s == 0) read_one(smem + cur, 1, r);
            if (r < kFrags && s == 1 && kLeft >= 1) read_one(smem + nxt, 0, r);
            if (r < kTileLoads && s == 1 && kLeft >= 3) issue_one(cur, r);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      cur = nxt;
    };
    issue(0);
    if (nk > 1) {
      advance(1);
      issue(1);
    }
    if (nk > 2) {
      advance(2);
      issue(2);
    }
    Base::zero(acc);
    // a zero of its own per accumulator: left to the compiler they are copies of one another,
    // made in front of every loop they enter
    pin(acc);
    if (nk > 2) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * kTileLoads) : "memory");
    else if (nk == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kTileLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kFrags; ++r) read_one(smem, 0, r);
    using Left0 = std::integral_constant<int, 0>;
    using Left1 = std::integral_constant<int, 1>;
    using Left2 = std::integral_constant<int, 2>;
    using Left3 = std::integral_constant<int, 3>;
    int k = 0;
    for (; k + 3 < nk; ++k) step(k, Left3{});
    if (k + 3 == nk) step(k++, Left2{});
    if (k + 2 == nk) step(k++, Left1{});
    step(k, Left0{});
    // as long as mfma_drain: the builtin's own distance is shorter, and the epilogue's
    // statements read accumulators without the compiler's knowledge of what wrote them
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 7");
    pin(acc);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
  }

  template <bool kAKMajor, bool kBKMajor>
  __device__ __forceinline__ void wide_loop(const Operand<T>& A, const Operand<T>& B, int k_begin,
                                            int k_end, Acc& acc, char* smem) const {
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    static_assert(!kColumnTail || (!kAKMajor && !kBKMajor), "column tails: K-contiguous operands");
    // K tiles of one pass
    const int pass_tiles = (k_end - k_begin) / kBK + (kColumnTail ? 1 : 0);
    const int nk = pass_tiles * kPasses;
    Loader la = make_loader<kAKMajor, kColumnTail>(A, k_begin, nk, lds0);
    Loader lb = make_loader<kBKMajor>(B, k_begin, nk, lds0 + kOperandBytes);
    // The place of a K tile among the passes, advanced one tile at a time.
    struct Place { int pass, tile; };
    auto next_place = [&](Place& at) {
      if (++at.tile == pass_tiles) {
        at.tile = 0;
        ++at.pass;
      }
    };
    // where a pass starts in an operand (no multiplication: the compiler forms 64-bit
    // products in vector registers, and the loads take their base from scalar ones)
    auto pass_start = [](const char* begin, int64_t plane, unsigned pass_planes, int pass) {
      const unsigned which = (pass_planes >> (4 * pass)) & 15u;
      return which == 0 ? begin : which == 1 ? begin + plane : begin + plane + plane;
    };
    Place load_at = {0, 0};
    if constexpr (kPlanes > 1) {
      la.next = pass_start(la.begin, la.plane, kPassPlaneA, 0);
      lb.next = pass_start(lb.begin, lb.plane, kPassPlaneB, 0);
    }
    // the loaders move on to K tile `k`, the next one
    auto advance = [&](int k) {
      if constexpr (kColumnTail) {
        const bool at_last = k == nk - 1;
        la.next = at_last ? la.last : la.next + la.step;
        lb.next += lb.step;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) la.off[j] = at_last ? la.last_off[j] : la.off[j];
      } else if constexpr (kPlanes == 1) {
        la.next = kAKMajor && k == nk - 1 ? la.last : la.next + la.step;
        lb.next = kBKMajor && k == nk - 1 ? lb.last : lb.next + lb.step;
      } else {
        next_place(load_at);
        if (load_at.tile != 0) {
          la.next += la.step;
          lb.next += lb.step;
        } else {
          la.next = pass_start(la.begin, la.plane, kPassPlaneA, load_at.pass);
          lb.next = pass_start(lb.begin, lb.plane, kPassPlaneB, load_at.pass);
        }
      }
    };
    const int ra = reader_base<kAKMajor>(wm);
    const int rb = reader_base<kBKMajor>(wn);

    // load number q (0..15) of the K tile the loaders stand at, into `stage`: even q -> A,
    // odd q -> B
    auto issue_one = [&](int stage, int q) {
      const unsigned s_off = (unsigned)(stage * kStageBytes) + (unsigned)((q >> 1) * 1024);
      if (q & 1) load_to_lds(lb.fill + s_off, lb.off[q >> 1], lb.next);
      else load_to_lds(la.fill + s_off, la.off[q >> 1], la.next);
    };
    V8 fa[kTM], fb[2][kTN];
    auto read_a = [&](int stage, int ks, int i) {
      fa[i] = read_frag<kAKMajor>(smem + stage * kStageBytes, ra, ks, i);
    };
    auto read_b = [&](int stage, int ks, int i) {
      fb[ks][i] = read_frag<kBKMajor>(smem + stage * kStageBytes + kOperandBytes, rb, ks, i);
    };

    // This wave's share of the touches: 64 lines of A (waves 0, 1) or B (waves 2, 3), in
    // the half of the tile's lines that the workgroup's neighbours leave to it.
    const bool touch_b = wave >= 2;
    const int line = (wave & 1) * 64 + lane +
                     (((touch_b ? A.row0 : B.row0) / kTile) & 1) * 128;
    const unsigned touch_off = touch_b ? line_offset<kBKMajor>(B, line) : line_offset<kAKMajor>(A, line);
    const int64_t touch_step = readfirstlane64(touch_b ? lb.step : la.step);
    const char* touch_base = reinterpret_cast<const char*>(
        readfirstlane64(reinterpret_cast<int64_t>(touch_b ? lb.begin : la.begin)));
    const unsigned touch_lds =
        __builtin_amdgcn_readfirstlane(lds0 + 2 * kStageBytes + (unsigned)wave * 256);
    // (a tail is small and in L2 already; the tile before it is touched again)
    const bool ragged = touch_b ? kBKMajor && k_end > B.k_full
                                : kColumnTail || (kAKMajor && k_end > A.k_full);
    const int touch_last = __builtin_amdgcn_readfirstlane(nk - 1 - (ragged ? 1 : 0));
    const unsigned touch_planes =
        __builtin_amdgcn_readfirstlane(touch_b ? kPassPlaneB : kPassPlaneA);
    const int64_t touch_plane = readfirstlane64(touch_b ? lb.plane : la.plane);
    Place touch_at = {0, 0};
    const char* touch_next = pass_start(touch_base, touch_plane, touch_planes, 0);
    auto next_touch = [&] {
      next_place(touch_at);
      touch_next = touch_at.tile != 0
                       ? touch_next + touch_step
                       : pass_start(touch_base, touch_plane, touch_planes, touch_at.pass);
    };
    if constexpr (kPlanes > 1) {
#pragma unroll
      for (int t = 0; t < kTouchAhead; ++t) next_touch();
    }
    auto touch_tile = [&](int k) {
      if constexpr (kPlanes == 1) {
        touch(touch_lds, touch_off, touch_base + (int64_t)min(k, touch_last) * touch_step);
      } else {
        // called for K tiles kTouchAhead, + 1, ...: past the last one the first again
        touch(touch_lds, touch_off, k < nk ? touch_next : touch_base);
        next_touch();
      }
    };
    // tiles_left: how many tiles follow (0, 1, or 2 for "two or more")
    auto step = [&](int k, auto tiles_left_tag, auto first_tag) {
      constexpr bool kHasNext = decltype(tiles_left_tag)::value >= 1;
      constexpr bool kHasTwo = decltype(tiles_left_tag)::value >= 2;
      constexpr bool kFirst = decltype(first_tag)::value;   // the first step sets the accumulators
      const int cur = k & 1;
      const int nxt = cur ^ 1;
      // fragments the allocator has moved between two steps with VALU copies: two wait
      // states before an MFMA may read them, which the compiler does not add for asm
      asm volatile("s_nop 1");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 16; ++g) {
        const int s = g >> 3;
        const int q = g & 7;
        if (kHasNext && s == 1 && q == 2) {
          // tile k+1 is complete and visible from here on; stage `cur` is free
          // (the one younger access is the touch of this step)
          asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
          __syncthreads();
          if (kHasTwo) advance(k + 2);
        }
#pragma unroll
        for (int t = 0; t < kTN; ++t) {
          if (kFirst && s == 0) Op::mma_set(fa[q], fb[s][t], acc.c[q][t]);
          else Op::mma(fa[q], fb[s][t], acc.c[q][t]);
          if (kHasNext && s == 0 && q == 4 && t == 3) touch_tile(k + kTouchAhead);
          // last A block of this slice
          if (q == 0 && t == 1) read_a(cur, s, kTM - 1);
          if (s == 0) {
            // slice 1 of this tile
            if (q < 2 && (t == 3 || t == 5)) read_b(cur, 1, 2 * q + (t == 5));
            if (q >= 2 && q < 6 && t == 5) read_b(cur, 1, q + 2);
            if (q >= 1 && t == 2) read_a(cur, 1, q - 1);
            if (kHasNext) {
              constexpr int kRest = 16 - kLoadsAfterBarrier;
              // two per group
              if ((t == 0 || t == 4) && 2 * q + (t == 4) < kRest)
                issue_one(nxt, kLoadsAfterBarrier + 2 * q + (t == 4));
            }
          } else if (kHasNext && q >= 2) {
            // slice 0 of the next tile
            if (q < 4 && (t == 1 || t == 3 || t == 5)) read_b(nxt, 0, (q - 2) * 3 + (t >> 1));
            if (q == 4 && (t == 1 || t == 3)) read_b(nxt, 0, 6 + (t >> 1));
            if (q < 4 && t == 7) read_a(nxt, 0, q - 2);
            if (q == 4 && t == 5) read_a(nxt, 0, 2);
            if (q == 4 && t == 7) read_a(nxt, 0, 3);
            if (q >= 5 && t == 3) read_a(nxt, 0, q - 1);
            if (kHasTwo && (t == 2 || t == 6) && 2 * (q - 2) + (t == 6) < kLoadsAfterBarrier)
              issue_one(cur, 2 * (q - 2) + (t == 6));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };

    // tile 0 entirely, then the first loads of tile 1 (la.next / lb.next always point at
    // the tile whose loads are being issued)
#pragma unroll
    for (int q = 0; q < 16; ++q) issue_one(0, q);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (nk > 1) {
      advance(1);
#pragma unroll
      for (int q = 0; q < kLoadsAfterBarrier; ++q) issue_one(1, q);
    }
#pragma unroll
    for (int r = 0; r < kTN; ++r) read_b(0, 0, r);
#pragma unroll
    for (int r = 0; r + 1 < kTM; ++r) read_a(0, 0, r);
    using Left0 = std::integral_constant<int, 0>;
    using Left1 = std::integral_constant<int, 1>;
    using Left2 = std::integral_constant<int, 2>;
    if (nk > 2) step(0, Left2{}, std::true_type{});
    else if (nk == 2) step(0, Left1{}, std::true_type{});
    else step(0, Left0{}, std::true_type{});
    int k = 1;
    for (; k + 2 < nk; ++k) step(k, Left2{}, std::false_type{});
    if (k + 2 == nk) step(k++, Left1{}, std::false_type{});
    if (k < nk) step(k, Left0{}, std::false_type{});
    mfma_drain(acc);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last touches have landed
    __syncthreads();
  }

  // The same with both operands K-contiguous.
  __device__ __forceinline__ void mainloop_set(const T* __restrict__ A, int64_t lda, int a_row0,
                                               int a_rows, const T* __restrict__ B, int64_t ldb,
                                               int b_row0, int b_rows, int k_begin, int k_end,
                                               Acc& acc, char* smem) const {
    const Operand<T> a = {A, lda, a_row0, a_rows};
    const Operand<T> b = {B, ldb, b_row0, b_rows};
    mainloop_ex<false, false>(a, b, k_begin, k_end, acc, smem);
  }
};

// 16-bit matrices as they are stored.
template <typename T_>
struct MfmaDirect4Engine : DirectToLdsEngine<T_, 1> {};

// The same for logits over hidden sizes that are no multiple of 64 (a multiple of 8, above 64):
// the last K tile of the first operand, the head, comes from a zero-padded copy of its last
// columns, and the second, the rows, is a copy padded with zeros to whole K tiles.  An engine
// of its own: the choice of the last tile's addresses costs the other up to 1.5 %.
template <typename T_>
struct ColumnTailEngine : DirectToLdsEngine<T_, 1, true> {};
// The engine of tiles with at most 32 * kTN rows of B beside E, where it has one (bool) and the
// LDS a launch takes that may run them all.
template <class E> constexpr bool kHasNarrowTiles = false;
template <typename T> constexpr bool kHasNarrowTiles<MfmaDirect4Engine<T>> = true;
template <typename T, int kTN> using NarrowEngine = DirectToLdsEngine<T, 1, false, kTN>;
template <class E>
constexpr int kLaunchSmemBytes =
    kHasNarrowTiles<E> ? (NarrowEngine<__bf16, 4>::kSmemBytes > E::kSmemBytes
                              ? NarrowEngine<__bf16, 4>::kSmemBytes
                              : E::kSmemBytes)
                       : E::kSmemBytes;

template <class E> constexpr bool kReadsColumnTails = false;
template <typename T> constexpr bool kReadsColumnTails<ColumnTailEngine<T>> = true;
// The engine that does so for engine E.
template <class E> struct ColumnTailOf { using type = E; };
template <typename T> struct ColumnTailOf<MfmaDirect4Engine<T>> { using type = ColumnTailEngine<T>; };

// Float32 matrices in three bf16 planes (tlce_split_f32.h): an operand's row holds its
// planes one after the other, so `ld` is the distance of two planes and a third of the
// distance of two rows.  The K loop runs once per pair of planes,
//   lo.hi  hi.lo  mid.mid  mid.hi  hi.mid  hi.hi
struct SplitF32Engine : DirectToLdsEngine<__bf16, 3> {};

}  // namespace tlce
