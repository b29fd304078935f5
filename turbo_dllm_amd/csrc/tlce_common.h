// Shared host/device helpers for the gfx950 fused linear cross-entropy library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <string.h>

#include <algorithm>

#include "../../include/tlce.h"

namespace tlce {

// ---------------------------------------------------------------- errors ----
// Thread-local message buffer behind tlce_last_error().  The reference raises
// through TORCH_CHECK (fused_linear_ce.cpp:107-111); here every entry point
// returns a code and leaves the text for the host binding to raise.
char* error_buffer();
int fail(const char* fmt, ...);

#define TLCE_HIP(expr)                                                        \
  do {                                                                        \
    hipError_t tlce_err__ = (expr);                                           \
    if (tlce_err__ != hipSuccess) {                                           \
      return ::tlce::fail("%s failed: %s (%s:%d)", #expr,                     \
                          hipGetErrorString(tlce_err__), __FILE__, __LINE__); \
    }                                                                         \
  } while (0)

#define TLCE_REQUIRE(cond, ...)           \
  do {                                    \
    if (!(cond)) {                        \
      return ::tlce::fail(__VA_ARGS__);   \
    }                                     \
  } while (0)

#define TLCE_LAUNCH_CHECK() TLCE_HIP(hipGetLastError())

// ----------------------------------------------------------------- sizes ----
static inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
static inline int64_t ceil_div(int64_t x, int64_t m) { return (x + m - 1) / m; }
static inline int64_t align256(int64_t x) { return round_up(x, 256); }

static inline int dtype_bytes(int dtype) { return dtype == TLCE_DTYPE_F32 ? 4 : 2; }

// Workgroups of a tile engine that the 256 CUs hold at once: the 256x256 engines take a CU
// each, the float32 MFMA engine (128x128 tiles) fits two on one.  The generic engine (64x64,
// 9 KiB of LDS) needs four on a CU to hide its loads: planned for one, its forward took 2.73
// instead of 1.18 ms (1000 bf16 rows, H = 1001, V = 16384).
__host__ __device__ static inline int resident_workgroups(int tile) {
  return tile == 64 ? 1024 : tile == 128 ? 512 : 256;
}

// Forward launch shape: token tiles x vocabulary splits workgroups, at most four whole
// rounds of 256 workgroups on a 256-CU MI355X.  Shared by the host plan and by the
// kernels that derive the plan from a row count that only the device knows.
//
// A split loops over ceil(n_vtiles / splits) tiles, so the launch lasts about
// rounds x (that + 1/8 for a workgroup's start and merge) tile times; of one to four
// rounds the cheapest is taken, ties going to fewer (longer loops keep the workgroups
// of an XCD in step).  Fewer than four splits leave an XCD's 32 workgroups more
// distinct operand strips than the usual 12, which costs time: 2 splits measured 9 %.
// Measured (ms, H = 4096, V = 151936; always four rounds -> this rule): 1610 rows
// 1.72 -> 1.60, 6357 rows 6.43 -> 5.62; 12000 rows over H = 2048, V = 65536 2.42 -> 2.37
// (three rounds); 32768 rows over V = 16384 keep 2.98 (one round of two splits 3.26).
constexpr int kTargetWorkgroups = 1024;
__host__ __device__ static inline int forward_vocab_splits(int n_ttiles, int n_vtiles,
                                                           int resident) {
  int pick = 1;
  int64_t best = -1;
  for (int rounds = 1; rounds <= kTargetWorkgroups / resident; ++rounds) {
    int splits = n_ttiles > 0 ? rounds * resident / n_ttiles : rounds * resident;
    splits = splits < 1 ? 1 : (splits < n_vtiles ? splits : n_vtiles);
    const int64_t launched = ((int64_t)n_ttiles * splits + resident - 1) / resident;
    const int64_t tiles = (n_vtiles + splits - 1) / splits;
    const int strips = splits >= 8   ? 100
                       : splits >= 4 ? 102
                       : splits == 3 ? 104
                       : splits == 2 ? 110
                                     : 133;
    const int64_t cost = launched * (8 * tiles + 1) * strips;
    if (best < 0 || cost < best) {
      best = cost;
      pick = splits;
    }
  }
  return pick;
}

// K splits of the grad_hidden contraction: `tiles` output tiles per panel, each a
// loop of `k_steps` K steps when unsplit; every split accumulates into a float32
// slab of its own (`slab_elems` elements), summed by the final cast.  Picks the
// count in [1, max_split] with the least estimated time, in eighths of a K step:
//   rounds of `resident` workgroups x (K steps per split + 8 for a tile's start and output)
//   + splits x the time the slab's write and its read by the final cast take.
// Up to 64 splits: 64 rows over H = 1024 are four tiles, whose K loop of 500 steps (V =
// 32000) ran on 64 CUs with at most 16 splits, 49 us; now 25.
// Ties go to fewer splits.  Integer arithmetic only (divisions in 32 bits: a K step is 64
// or 32 wide): the host plan and the kernels that re-plan for a row count known on the
// device must agree.
constexpr int kMaxKSplits = 64;
// The estimate for `ks` splits; per_slab: k_split_slab_cost.
__host__ __device__ static inline int64_t k_split_cost(int64_t tiles, int ks, int64_t k_steps,
                                                       int64_t per_slab, int resident) {
  const int shift = 31 - __builtin_clz(resident);
  const int64_t rounds = (tiles * ks + resident - 1) >> shift;
  const int64_t steps = ((uint32_t)k_steps + (uint32_t)ks - 1) / (uint32_t)ks;
  return rounds * 8 * (steps + 8) + ks * per_slab;
}
__host__ __device__ static inline int64_t k_split_slab_cost(int64_t slab_elems) {
  return (slab_elems >> 17) > 1 ? (slab_elems >> 17) : 1;
}
static inline int grad_hidden_k_splits(int64_t tiles, int max_split, int64_t k_steps,
                                       int64_t slab_elems, int resident = 256) {
  const int64_t per_slab = k_split_slab_cost(slab_elems);
  int pick = 1;
  int64_t best = -1;
  for (int ks = 1; ks <= max_split; ++ks) {
    const int64_t cost = k_split_cost(tiles, ks, k_steps, per_slab, resident);
    if (best < 0 || cost < best) {
      best = cost;
      pick = ks;
    }
  }
  return pick;
}

constexpr int kXcds = 8;  // MI355X: 8 accelerator dies, workgroups dealt round-robin

// ------------------------------------------------------------- device -------
#define TLCE_LOG2E 1.4426950408889634f
#define TLCE_LN2 0.6931471805599453f

// Workgroups are dealt to the 8 XCDs round-robin by blockIdx; each XCD has its
// own L2.  Map the hardware block id to a logical id so that one XCD works on
// a contiguous range of logical ids (launch grids are multiples of 8).
__device__ __forceinline__ int xcd_logical_block(int bid, int nblocks) {
  const int per = nblocks / kXcds;
  return (bid % kXcds) * per + (bid / kXcds);
}

// Rows of a call whose row count lives on the device: `m` is then the
// capacity the launch was sized for and *m_dev (clamped to [0, m]) the real
// count.  m_dev == null: m itself.
__device__ __forceinline__ int effective_rows(int m, const int64_t* m_dev) {
  if (m_dev == nullptr) return m;
  const int64_t c = *m_dev;
  return c < 0 ? 0 : (c < (int64_t)m ? (int)c : m);
}

// Rows of a block of `cap` rows that starts at row `offset` of a matrix whose real
// row count is on the device (null: all `cap`).
__device__ __forceinline__ int effective_block_rows(int cap, const int64_t* m_dev, int64_t offset) {
  if (m_dev == nullptr) return cap;
  const int64_t c = *m_dev - offset;
  return c < 0 ? 0 : (c < (int64_t)cap ? (int)c : cap);
}

// Logical block id when only the first `tiles` of the launched workgroups have
// work (the launch was sized for more rows than there are): the same mapping a
// launch of round_up(tiles, 8) workgroups would get; -1 for the others.
__device__ __forceinline__ int xcd_logical_block_of(int bid, int tiles) {
  const int total = (tiles + kXcds - 1) / kXcds * kXcds;
  if (bid >= total) return -1;
  const int logical = xcd_logical_block(bid, total);
  return logical < tiles ? logical : -1;
}

// Grouped tile order: consecutive logical ids walk a group of at most `group` tiles
// along i, then step j, so the ~32 workgroups resident on one XCD cover a group x
// (32/group) block of tiles and share both operands through that XCD's L2.  The groups
// are balanced: ceil(ni / group) groups whose sizes differ by at most one (13 tiles in
// groups of at most 4: 4, 3, 3, 3 instead of 4, 4, 4, 1; a group of one tile has its 32
// workgroups fetch 33 strips instead of 12: 9 token tiles in groups of 4, 4, 1 took the
// forward 1.51 ms against 1.28 balanced, 5 hidden tiles grad_weight 0.65 against 0.59).
__device__ __forceinline__ void grouped_tile(int logical, int ni, int nj, int group,
                                             int* ti, int* tj) {
  const int n_groups = (ni + group - 1) / group;
  const int base = ni / n_groups, extra = ni % n_groups;   // the first `extra` groups hold base + 1
  const int big = (base + 1) * nj;
  int first, gsize, within;
  if (logical < extra * big) {
    const int g = logical / big;
    gsize = base + 1;
    first = g * gsize;
    within = logical - g * big;
  } else {
    const int rest = logical - extra * big;
    const int g = rest / (base * nj);
    gsize = base;
    first = extra * (base + 1) + g * base;
    within = rest - g * base * nj;
  }
  *ti = first + within % gsize;
  *tj = within / gsize;
}

// Whether the eighths of a launch ordered by groups of four tiles begin at the same j (xcd_tile).
__host__ __device__ static inline bool xcd_aligned(int ni) {
  const int groups = (ni + 3) / 4;
  return (ni % 4) == 0 && (groups <= 2 || (groups % 4) == 0);
}

// Which output tile a workgroup of an ni x nj tile contraction takes (`strip` = bytes of
// one operand strip of 256 rows over the whole K range); false: none.  The launch has
// xcd_grid(ni * nj) workgroups.
//
// L2 is shared by an XCD's ~32 resident workgroups, the 256 MiB last-level cache by all
// XCDs, and what a CU cannot get from either costs HBM time and power.  Two orders:
//   by groups : a group of four tiles along i, all of j, then the next group; XCD x takes
//               the x-th eighth.  When the eighths begin at the same j (whole groups per
//               XCD, or a half or a quarter of one), the XCDs stream the j strips in step
//               and fetch each from HBM once.
//   by blocks : eight tiles along j with all of i (in groups of four), then the next
//               eight; each XCD reads its own j strips from HBM once and again, for the
//               further groups, from the last-level cache, where all the i strips stay.
//               Four tiles along j when only those fit beside the i strips.
// By groups where the eighths are aligned, unless the strips are so short that the cache
// holds them anyway.  The two limits, on the strips that eight tiles per XCD and all of i
// make, are where the measured pairs cross (ms, bf16, V = 151936, H = 4096 unless stated;
// E: exponentiated logits, W: grad_weight of 16 or, unaligned, of 15 hidden tiles, H = 3840).
// By groups / by blocks of eight, aligned:
//   40 MiB  E 4096 rows, H = 1024    1.36 / 1.30      90 MiB  E 4096, H = 2304   2.23 / 2.29
//   50 MiB  W 1280 rows              1.49 / 1.40     100 MiB  W 2560             2.53 / 2.55
//   60 MiB  E 4096, H = 1536         1.68 / 1.66     120 MiB  E 8192, H = 2560   4.81 / 4.89
//   70 MiB  W 1792                   1.88 / 1.88     144 MiB  E 8192, H = 3072   5.57 / 5.65
//   80 MiB  E 4096, H = 2048         2.04 / 2.04     192 MiB  E 8192             7.26 / 7.39
//   96 MiB  E 8192, H = 2048         3.98 / 3.99     320 MiB  W 8192             7.35 / 7.65
// By groups / blocks of eight / blocks of four, unaligned:
//  165 MiB  E 6144 rows, H = 3840    5.31 / 5.29 / 5.28
//  198 MiB  W 5120                   4.50 / 4.42 / 4.40
//  206 MiB  E 8448, H = 4352         8.58 / 8.18 / 8.25
//  242 MiB  E 8448, H = 5120        10.08 / 9.73 / 9.66
//  316 MiB  W 8192                   7.27 / 7.21 / 6.98
//  326 MiB  W 8448                   7.48 / 7.40 / 7.16
// (past 224 MiB for blocks of four too, eight are taken: 12288 rows W 10.71 / 10.87 / 10.65,
// grad_hidden over the whole vocabulary 10.61 / 10.87 / 10.99, in 15 hidden tiles of 8448
// rows 7.65 / 7.12 / 7.22)
__device__ __forceinline__ bool xcd_tile(int bid, int ni, int nj, int64_t strip, int* ti,
                                         int* tj) {
  const int64_t total = (int64_t)ni * nj;
  const int64_t kib = strip >> 10;
  if (xcd_aligned(ni) && (8 * 8 + ni) * kib > 84 * 1024) {
    const int logical = xcd_logical_block_of(bid, (int)total);
    if (logical < 0) return false;
    grouped_tile(logical, ni, nj, 4, ti, tj);
    return true;
  }
  const int xcd = bid % kXcds;
  const int first = (int)(xcd * total / kXcds), last = (int)((xcd + 1) * total / kXcds);
  int idx = first + bid / kXcds;
  if (idx >= last) return false;
  const bool narrow = (8 * 8 + ni) * kib > 224 * 1024 && (8 * 4 + ni) * kib <= 224 * 1024;
  const int width = narrow ? 4 : 8;
  const int blocks = (nj + width - 1) / width;   // balanced: `extra` of them one tile wider
  const int base = nj / blocks, extra = nj % blocks;
  const int wide = extra * (base + 1) * ni;      // tiles in the wider blocks
  int w = base + 1, j0 = 0;
  if (idx >= wide) {
    idx -= wide;
    w = base;
    j0 = extra * (base + 1);
  }
  const int b = idx / (ni * w);
  grouped_tile(idx - b * ni * w, ni, w, 4, ti, tj);
  *tj += j0 + b * w;
  return true;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// tanh(x) = 1 - 2 / (1 + e^{2x}); saturates cleanly to +-1 for large |x|.
__device__ __forceinline__ float fast_tanh(float x) {
  const float e = fast_exp2(x * (2.0f * TLCE_LOG2E));
  return 1.0f - 2.0f * fast_rcp(1.0f + e);
}

// Elementwise math by engine.  The float32 engine (float32 inputs, held to the
// reference's 2e-5 bars) takes the library routines: fast_tanh loses relative
// accuracy for small arguments (1 - 2 / (1 + e) cancels), which the soft cap's
// derivative then carries into the gradient.  The 16-bit engines take the
// hardware approximations, whose error is far below the rounding of their inputs.
template <bool kPrecise>
__device__ __forceinline__ float exp2_of(float x) {
  if constexpr (kPrecise) return exp2f(x);
  else return fast_exp2(x);
}
template <bool kPrecise>
__device__ __forceinline__ float log2_of(float x) {
  if constexpr (kPrecise) return log2f(x);
  else return fast_log2(x);
}
template <bool kPrecise>
__device__ __forceinline__ float tanh_of(float x) {
  if constexpr (kPrecise) return tanhf(x);
  else return fast_tanh(x);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename T>
__device__ __forceinline__ float to_float(T x) { return static_cast<float>(x); }
template <typename T>
__device__ __forceinline__ T from_float(float x) { return static_cast<T>(x); }

// Host-side launch grid: a multiple of 8 so xcd_logical_block is a bijection.
static inline int xcd_grid(int64_t tiles) { return (int)round_up(tiles, kXcds); }

}  // namespace tlce
