// Host scheduler of the fused linear cross-entropy for gfx950: tile plans,
// workspace layouts, kernel launches and the per-objective launch sequences,
// templated on a tile engine.
//
// Replaces fused_linear_ce_forward_cuda / fused_linear_ce_backward_cuda
// (dllm_parallel/core/csrc/fused_linear_ce/fused_linear_ce_cuda.cu:898-989,
// :991-1172).  Where the reference loops over ~1K-row blocks and round-trips
// float32 logits through memory three times per block, this scheduler
//   forward : one launch of the online-softmax tile kernel (+ a per-row merge);
//   backward: loops over vocabulary panels; per panel one launch recomputes the
//             logits tiles and writes the dtype-rounded logit gradients of the
//             panel, one contraction accumulates grad_hidden in float32 and
//             one writes the panel's rows of grad_weight, complete, in dtype.
// Nothing here allocates or synchronises.
//
// The launch sequences are instantiated once per engine, each in a translation
// unit of its own (tlce_engine_*.hip), so that the library builds in parallel;
// the C ABI (tlce_linear_ce.hip) sees them as extern templates.
#pragma once

#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <vector>

#include "tlce_common.h"
#include "tlce_engine_f32.h"
#include "tlce_engine_mfma.h"
#include "tlce_engine_simt.h"
#include "tlce_kernels.h"

namespace tlce {

// ------------------------------------------------------------- profiling ----
// Optional per-kernel-class timing with HIP events on the caller's stream
// (tlce_profile_begin / tlce_profile_end).  Off by default; when off a launch
// costs one thread-local pointer test.  One profiling session per thread.
enum KernelClass {
  kClassForwardStats = 0,
  kClassCombine = 1,
  kClassGradLogits = 2,
  kClassGradHidden = 3,
  kClassGradWeight = 4,
  kClassTranspose = 5,
  kClassOther = 6,
  kClassExpPanel = 7,
  kNumClasses = 8
};

struct Profiler {
  struct Record { int cls; hipEvent_t start, stop; };
  std::vector<Record> records;
};
extern thread_local Profiler* g_profiler;   // defined beside the C ABI

struct ScopedTimer {
  Profiler* prof;
  hipStream_t stream;
  hipEvent_t start = nullptr, stop = nullptr;
  int cls;
  ScopedTimer(int cls_, hipStream_t s) : prof(g_profiler), stream(s), cls(cls_) {
    if (!prof) return;
    if (hipEventCreate(&start) != hipSuccess || hipEventCreate(&stop) != hipSuccess) {
      prof = nullptr;
      return;
    }
    (void)hipEventRecord(start, stream);
  }
  ~ScopedTimer() {
    if (!prof) return;
    (void)hipEventRecord(stop, stream);
    prof->records.push_back({cls, start, stop});
  }
};

constexpr int64_t kDefaultPanelBytes = 1ll << 30;

struct Plan {
  int64_t v;    // vocabulary rows
  int engine;   // 3 = float32 MFMA, 2 = direct-to-LDS MFMA, 1 = register-staged MFMA, 0 = generic
  bool kmajor;  // gradient contractions read K-major operands in place
  int64_t column_tail;  // not 0: the logits contractions read copies of the operands
                        // (launch_column_tails), hidden's with rows of this length
  int tile;
  int bk;
  int64_t mp, vp;
  int n_ttiles, n_vtiles, n_htiles;
  int nsplit;         // forward vocabulary splits
  int64_t vc;         // panel columns
  int n_panels;
  int dh_ksplit;
  int dh_max_ksplit;  // upper bound of the rule that chose dh_ksplit
  int64_t dh_slab_rows;   // rows of all K-split slabs together
};

inline int engine_class(int64_t h, int dtype) {
  if (dtype == TLCE_DTYPE_F32) return (h % 4) == 0 ? 3 : 0;
  if ((h % 8) != 0) return 0;
  return (h % 64) == 0 ? 2 : 1;
}

// Rows of all K-split slabs of a grad_hidden contraction together.  A row count on the device may
// leave fewer tiles, and more splits of them, than n_ttiles have: slabs for one round of workgroups
// (64 MiB at most), so that it gets the splits of a call with that many rows where they make one.
// 2240 of 3200 rows, H = 2112 (81 of 117 tiles) take three splits and not the plan's two.
inline int64_t k_split_slab_rows(int ksplit, int max_split, int n_ttiles, int n_htiles, int tile) {
  const int64_t round = std::min<int64_t>(ceil_div(resident_workgroups(tile), n_htiles),
                                          (int64_t)n_ttiles * max_split);
  return std::max((int64_t)ksplit * n_ttiles, round) * tile;
}

// Whether the caller has scratch for copies of operands (column tails), and what for.
enum ColumnTails { kNoColumnTails, kForwardTails, kBackwardTails };

inline Plan make_plan(int64_t m, int64_t h, int64_t v, int dtype, bool weight_grad,
               int64_t panel_bytes, int max_engine = 3, ColumnTails tails = kNoColumnTails) {
  Plan p;
  p.v = v;
  p.column_tail = 0;
  // 16-bit inputs: 2: four-wave direct-to-LDS MFMA (h % 64 == 0), 1: register-staged MFMA
  // (h % 8 == 0); float32: 3: float32 MFMA (h % 4 == 0); 0: generic float32-FMA tiles
  p.engine = std::min(engine_class(h, dtype), max_engine);
  // a float32 vocabulary that one generic tile holds would leave most of a 128x128 tile
  // and of its matrix instructions empty (both take about 10 us there)
  if (p.engine == 3 && v < 64) p.engine = 0;
  // Hidden sizes that are multiples of 8 but not of 64: the direct engine takes the last K tile
  // of the head from a zero-padded copy of its last columns and hidden from a padded copy
  // (callers with scratch for them).  Forward / both directions in us, staged -> direct:
  //   4096 rows, H = 2040, V = 65536   1203 -> 1001 / 5100 -> 3688  (H = 2048: 820 / 2550,
  //                                    from three contractions and aligned rows of the head)
  //   300 rows, H = 1000, V = 16384    89 -> 83 / 291 -> 253
  //   70 rows, H = 5000, V = 32000     242 -> 188 / 995 -> 636
  // Short rows are mostly tail and the copies' launch is part of small calls: forward at
  // H = 72, 4096 rows, V = 32000 108 -> 117; H = 136, 2048 rows, V = 1024 72 -> 77 (2 to 3 us of
  // a forward alone also at H = 264 to 728).
  // Over few words the copy of many rows costs more than the contraction gains, and what
  // remains of it there is the gradient of the head.  65536 rows, staged -> direct, forward /
  // its backward under a frozen head / both directions with a trainable one:
  //   H = 1000, V = 512    175 -> 227 / 343 -> 365 / 2439 -> 1877     V = 1024  248 -> 279 / 504 -> 473
  //   H = 1992, V = 256    191 -> 340 / 492 -> 562 / 2726 -> 2476     V = 2048  681 -> 696 / 1492 -> 1255
  const bool few_rows = m <= 8192 && m * h <= (1ll << 25);
  const bool enough_words = few_rows || (tails == kForwardTails ? v >= 2048
                                                                : weight_grad || v >= 1024);
  if (tails != kNoColumnTails && p.engine == 1 && h >= 256 && m > 64 && m * v >= (1ll << 21) &&
      enough_words) {
    p.engine = 2;
    p.column_tail = round_up(h, 64);
  }
  // The direct and the float32 engine read weight, hidden and the logit-gradient panel
  // in their stored form for the gradient contractions (no transposed copies).  The
  // direct one takes whole 64-row K slabs: of a last, incomplete slab of weight or
  // hidden a zero-padded copy is made (launch_k_tail).
  p.kmajor = p.engine >= 2;
  p.tile = p.engine == 3 ? 128 : p.engine ? 256 : 64;
  p.bk = p.engine == 3 ? 32 : p.engine ? 64 : 16;
  const int64_t mm = std::max<int64_t>(m, 1);
  p.mp = round_up(mm, p.tile);
  p.vp = round_up(v, p.tile);
  p.n_ttiles = (int)(p.mp / p.tile);
  p.n_vtiles = (int)(p.vp / p.tile);
  p.n_htiles = (int)ceil_div(h, p.tile);
  // forward: token tiles x vocabulary splits workgroups, whole rounds of 256
  p.nsplit = forward_vocab_splits(p.n_ttiles, p.n_vtiles, resident_workgroups(p.tile));
  if (panel_bytes <= 0) panel_bytes = kDefaultPanelBytes;
  const int64_t col_bytes = p.mp * dtype_bytes(dtype) * ((weight_grad && !p.kmajor) ? 2 : 1);
  int64_t tiles_per_panel = std::max<int64_t>(1, panel_bytes / col_bytes / p.tile);
  tiles_per_panel = std::min<int64_t>(tiles_per_panel, p.n_vtiles);
  // A panel of 16*k vocabulary tiles gives the grad_weight launch (tiles x
  // n_htiles workgroups) and the logit-gradient launch (tiles x n_ttiles) whole
  // waves of 256 workgroups at the usual head sizes; the last panel takes the
  // remainder.  Small problems fall back to equal panels.
  if (tiles_per_panel >= 16 && tiles_per_panel < p.n_vtiles) {
    tiles_per_panel = tiles_per_panel / 16 * 16;
    p.vc = tiles_per_panel * p.tile;
  } else {
    p.n_panels = (int)ceil_div(p.n_vtiles, tiles_per_panel);
    p.vc = ceil_div(p.n_vtiles, p.n_panels) * p.tile;  // balanced panels
  }
  p.n_panels = (int)ceil_div(p.vp, p.vc);
  // grad_hidden: n_ttiles x n_htiles tiles per panel.  When that is not close
  // to whole waves of 256 workgroups, split K (each split accumulates into its
  // own float32 slab, summed by the final cast) by the factor with the least
  // estimated time (grad_hidden_k_splits).
  p.dh_ksplit = 1;
  p.dh_max_ksplit = 1;
  if (p.engine) {
    p.dh_max_ksplit = (int)std::max<int64_t>(1, std::min<int64_t>(kMaxKSplits, p.vc / p.bk / 8));
    p.dh_ksplit = grad_hidden_k_splits((int64_t)p.n_ttiles * p.n_htiles, p.dh_max_ksplit,
                                       p.vc / p.bk, p.mp * h, resident_workgroups(p.tile));
  }
  p.dh_slab_rows = k_split_slab_rows(p.dh_ksplit, p.dh_max_ksplit, p.n_ttiles, p.n_htiles, p.tile);
  return p;
}

// What the masked-token loss adds to the plain operator
// (distributed_block_diffusion_loss, nemotron/model.py:2084-2151): the output
// multiplier applied to the logits instead of to a copy of the hidden states,
// per-row loss weights, the weighted loss sum, and a row count that stays on
// the device (row_count != null: m is the capacity every launch is sized for).
struct RowOptions {
  float logit_scale = 1.0f;
  const float* token_weights = nullptr;   // [m] float32, compacted order
  const int64_t* row_count = nullptr;     // device int64
  float* weighted_sum = nullptr;          // forward: [1] float32 out
  // the head and its gradient are stored [h, v] (weight_dim_first of the reference's
  // extension, fused_linear_ce.cpp:104,121) and are read / written in place
  bool weight_dim_first = false;
  KeptLogits kept;                        // written by the forward, read by the backward
};

// A [h, v] head is taken in place by the engine with K-major operand loaders, for
// vocabularies made of whole 64-row K slabs.
inline bool dim_first_in_place(int64_t h, int64_t v, int dtype) {
  return engine_class(h, dtype) == 2 && (v % 64) == 0;
}

// How many of the first vocabulary tiles' products a recomputing cross entropy's forward keeps
// for its backward within `budget` bytes (0: none).  A kept logit costs 4 bytes written beside
// the statistics, which passes under the contraction, and 4 read in the place of 2 h operations.
// Forward and backward with a trainable head in us, recomputed / kept, bf16:
//   8192 rows, H =  768, V =  65537   3033 /  3275      1000, H =  768, V =  50001    438 /  419
//   8192 rows, H = 1024, V = 151937   8243 /  8116      2741, H = 1024, V =  32003    708 /  678
//   4096 rows, H = 1280, V =  50001   1731 /  1592      8192, H = 1536, V = 151937  11669 / 10744
//   2741 rows, H = 2048, V =  32003   1288 /  1130       500, H = 2048, V =  32003    366 /  327
//    300 rows, H = 3072, V =  65537    864 /   691      4096, H = 4096, V = 151937  14407 / 11856
//   4096 rows, H = 2040, V =  65536   3581 /  3058      16384, H = 4096, V = 151936 55836 / 45655
constexpr int64_t kKeptTileBytes = (int64_t)kKeptTileFloats * 4;
constexpr int64_t kKeepMinHidden = 1024;
inline int64_t kept_vocab_tiles(int64_t m, int64_t h, int64_t v, int dtype, bool bias,
                                int64_t budget) {
  if (m <= 0 || bias || dtype == TLCE_DTYPE_F32 || h < kKeepMinHidden) return 0;
  const Plan p = make_plan(m, h, v, dtype, false, 0, 3, kBackwardTails);
  const Plan f = make_plan(m, h, v, dtype, false, 0, 3, kForwardTails);
  if (p.engine != 2 || f.engine != 2) return 0;
  return std::max<int64_t>(0, std::min<int64_t>(p.n_vtiles, budget / (kKeptTileBytes * p.n_ttiles)));
}
inline KeptLogits kept_logits(const Plan& p, void* tiles, int64_t bytes) {
  KeptLogits k;
  k.tiles = static_cast<float*>(tiles);
  k.t_tiles = p.n_ttiles;
  if (tiles != nullptr && p.n_ttiles > 0)
    k.v_tiles = (int)std::min<int64_t>(p.n_vtiles, bytes / (kKeptTileBytes * p.n_ttiles));
  return k;
}

// Bytes of what launch_column_tails writes: the copy of weight's last columns [vp, 64], then
// that of hidden [mp, column_tail].
inline int64_t column_tail_bytes(const Plan& p) {
  return p.column_tail != 0 ? (p.vp * 64 + p.mp * p.column_tail) * 2 : 0;
}

struct ForwardLayout {
  int64_t part_max, part_sum, weighted, tails, total;
};
// dynamic_rows: the partials must fit whatever plan the kernels derive from a
// device-side row count <= m (at most kTargetWorkgroups tiles, or one split of
// all token tiles); weighted: room for the per-row weighted losses.
inline ForwardLayout forward_layout(const Plan& p, bool dynamic_rows = false,
                                    bool weighted = false) {
  ForwardLayout l;
  int64_t floats = (int64_t)p.nsplit * p.mp;
  if (dynamic_rows) floats = std::max<int64_t>((int64_t)kTargetWorkgroups * p.tile, p.mp);
  const int64_t part = align256(floats * 4);
  l.part_max = 0;
  l.part_sum = part;
  l.weighted = 2 * part;
  l.tails = 2 * part + (weighted ? align256(p.mp * 4) : 0);
  l.total = l.tails + column_tail_bytes(p);
  return l;
}

struct BackwardLayout {
  int64_t scale, acc32, wt, ht, g, gt, tails, total;
};
// Bytes of the zero-padded copy of a 16-bit [rows, h] matrix's last K slab that a
// direct-engine contraction over its rows needs (none: all slabs are whole).
inline int64_t k_tail_bytes(int64_t rows, int64_t h) {
  return rows % 64 != 0 ? align256(64 * h * 2) : 0;
}

// wt / ht / gt are transposed copies on the path of the engines without K-major
// operands; on the direct engine's path wt and ht are the K tails of weight and hidden.
inline BackwardLayout backward_layout(const Plan& p, int64_t m, int64_t h, int dtype, bool weight_grad) {
  BackwardLayout l;
  const int64_t es = dtype_bytes(dtype);
  int64_t off = 0;
  l.scale = off; off += align256(p.mp * 4);
  l.acc32 = off; off += align256(p.dh_slab_rows * h * 4);   // one slab per K split
  const bool direct = p.engine == 2;
  l.wt = off;    off += direct ? k_tail_bytes(p.v, h) : p.kmajor ? 0 : align256(h * p.vp * es);
  l.ht = off;
  if (weight_grad) off += direct ? k_tail_bytes(m, h) : p.kmajor ? 0 : align256(h * p.mp * es);
  l.g = off;     off += align256(p.mp * p.vc * es);
  l.gt = off;    off += (weight_grad && !p.kmajor) ? align256(p.vc * p.mp * es) : 0;
  l.tails = off; off += column_tail_bytes(p);
  l.total = off;
  return l;
}

// Kernels with more than 64 KiB of dynamic LDS need the limit raised once per
// kernel and device; `done` is the calling site's per-device record.
constexpr int kMaxDevices = 64;
struct LdsOptIn {
  std::atomic<bool> done[kMaxDevices] = {};
};

template <typename K>
int enable_large_lds(K kernel, int bytes, LdsOptIn& state) {
  if (bytes <= 64 * 1024) return 0;
  int device = 0;
  TLCE_HIP(hipGetDevice(&device));
  const bool tracked = device >= 0 && device < kMaxDevices;
  if (tracked && state.done[device].load(std::memory_order_acquire)) return 0;
  TLCE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  if (tracked) state.done[device].store(true, std::memory_order_release);
  return 0;
}

inline int validate_common(const void* hidden, const void* weight, int64_t m, int64_t h, int64_t v,
                    int dtype) {
  TLCE_REQUIRE(dtype == TLCE_DTYPE_F32 || dtype == TLCE_DTYPE_F16 || dtype == TLCE_DTYPE_BF16,
               "unsupported dtype code %d", dtype);
  TLCE_REQUIRE(m >= 0 && h > 0 && v > 0, "bad shape m=%lld h=%lld v=%lld", (long long)m,
               (long long)h, (long long)v);
  TLCE_REQUIRE(m < (1ll << 30) && h < (1ll << 30) && v < (1ll << 30),
               "shape exceeds 32-bit tile indexing");
  TLCE_REQUIRE(weight != nullptr && (hidden != nullptr || m == 0), "null input pointer");
  TLCE_REQUIRE(((uintptr_t)hidden & 15) == 0 && ((uintptr_t)weight & 15) == 0,
               "hidden and weight must be 16-byte aligned");
  return 0;
}

// ---------------------------------------------------------------- launches --
template <class E, bool kSoftcap, bool kBias, bool kWDimFirst = false>
int launch_forward_variant(const Plan& p, const ForwardArgs& a, hipStream_t stream) {
  static LdsOptIn lds;
  if (int rc = enable_large_lds(lce_forward_stats_kernel<E, kSoftcap, kBias, kWDimFirst>,
                                E::kSmemBytes, lds))
    return rc;
  // with a device-side row count: the most tiles any row count <= m can plan
  const int64_t tiles =
      a.m_dev == nullptr
          ? (int64_t)p.n_ttiles * p.nsplit
          : std::min<int64_t>((int64_t)p.n_ttiles * p.n_vtiles,
                              std::max<int64_t>(kTargetWorkgroups, p.n_ttiles));
  const int grid = xcd_grid(tiles);
  ScopedTimer timer(kClassForwardStats, stream);
  lce_forward_stats_kernel<E, kSoftcap, kBias, kWDimFirst>
      <<<grid, E::kThreads, E::kSmemBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

template <class E>
int launch_forward(const Plan& p, const ForwardArgs& a, hipStream_t stream) {
  const bool softcap = a.softcap > 0.0f, bias = a.bias != nullptr;
  if (softcap && bias) return launch_forward_variant<E, true, true>(p, a, stream);
  if (softcap) return launch_forward_variant<E, true, false>(p, a, stream);
  if (bias) return launch_forward_variant<E, false, true>(p, a, stream);
  return launch_forward_variant<E, false, false>(p, a, stream);
}

// The engine that takes a head stored [h, v] in place (dim_first_in_place).
template <class E>
constexpr bool kTakesDimFirst = E::kHasKMajor && sizeof(typename E::T) == 2;

// The same over a head stored [h, v].
template <class E>
int launch_forward_dim_first(const Plan& p, const ForwardArgs& a, hipStream_t stream) {
  if constexpr (kTakesDimFirst<E>) {
    const bool softcap = a.softcap > 0.0f, bias = a.bias != nullptr;
    if (softcap && bias) return launch_forward_variant<E, true, true, true>(p, a, stream);
    if (softcap) return launch_forward_variant<E, true, false, true>(p, a, stream);
    if (bias) return launch_forward_variant<E, false, true, true>(p, a, stream);
    return launch_forward_variant<E, false, false, true>(p, a, stream);
  } else {
    return fail("this engine cannot read a [h, v] head in place");
  }
}

template <class E, bool kSoftcap, bool kBias, bool kWDimFirst = false>
int launch_grad_logits_variant(const GradLogitsArgs& a, hipStream_t stream) {
  static LdsOptIn lds;
  if (int rc = enable_large_lds(lce_grad_logits_panel_kernel<E, kSoftcap, kBias, kWDimFirst>,
                                (kGradLogitsLdsBytes<E, kBias>), lds))
    return rc;
  const int grid = xcd_grid((int64_t)a.n_ttiles * a.n_ptiles);
  ScopedTimer timer(kClassGradLogits, stream);
  lce_grad_logits_panel_kernel<E, kSoftcap, kBias, kWDimFirst>
      <<<grid, E::kThreads, (kGradLogitsLdsBytes<E, kBias>), stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

// The logit-gradient panel over a head stored [h, v].
template <class E>
int launch_grad_logits_dim_first(const GradLogitsArgs& a, hipStream_t stream) {
  if constexpr (kTakesDimFirst<E>) {
    const bool softcap = a.softcap > 0.0f, bias = a.bias != nullptr;
    if (softcap && bias) return launch_grad_logits_variant<E, true, true, true>(a, stream);
    if (softcap) return launch_grad_logits_variant<E, true, false, true>(a, stream);
    if (bias) return launch_grad_logits_variant<E, false, true, true>(a, stream);
    return launch_grad_logits_variant<E, false, false, true>(a, stream);
  } else {
    return fail("this engine cannot read a [h, v] head in place");
  }
}

template <typename T>
int launch_grad_from_kept(const GradLogitsArgs& a, const KeptLogits& kept, hipStream_t stream) {
  const int64_t grid = (int64_t)kept.t_tiles * a.n_ptiles * 4;   // quarters of tiles
  ScopedTimer timer(kClassGradLogits, stream);
  if (a.softcap > 0.0f)
    lce_grad_from_kept_kernel<T, true><<<(int)grid, 256, 0, stream>>>(a, kept);
  else
    lce_grad_from_kept_kernel<T, false><<<(int)grid, 256, 0, stream>>>(a, kept);
  TLCE_LAUNCH_CHECK();
  return 0;
}

template <class E>
int launch_grad_logits(const GradLogitsArgs& a, hipStream_t stream) {
  const bool softcap = a.softcap > 0.0f, bias = a.bias != nullptr;
  if (softcap && bias) return launch_grad_logits_variant<E, true, true>(a, stream);
  if (softcap) return launch_grad_logits_variant<E, true, false>(a, stream);
  if (bias) return launch_grad_logits_variant<E, false, true>(a, stream);
  return launch_grad_logits_variant<E, false, false>(a, stream);
}

// Tiles along j of a chunk of an unsplit contraction of ni x nj tiles (GemmArgs::j_chunk), or 0:
// a chunk is one round of workgroups, so that the second operand's strips are read in one round
// only and by few XCDs.  In one piece the two rounds of an unaligned launch (xcd_tile) both go
// over all of j, XCDs drift apart over a long K loop, and what they share is fetched again.  Taken
// where the chunks need no more rounds than the whole; aligned launches gain nothing (512 tiles of
// 8192 rows, H = 4096, V = 151936: 7.12 / 7.11 ms).  In one piece / in chunks, grad_hidden, ms:
//   8704 rows, H = 3840, V = 262144   14.03 / 12.20       9216, H = 3584, V = 65536   3.00 / 2.97
//   8212 rows, H = 3840, V = 262144   13.15 / 12.68      12288, H = 3840, V = 65536   4.66 / 4.55
//   8448 rows, H = 3840, V = 151936    6.93 / 6.72       11776, H = 2816, V = 65536   3.00 / 3.00
inline int round_chunk(int ni, int nj, int tile) {
  const int resident = resident_workgroups(tile);
  const int64_t rounds = ceil_div((int64_t)ni * nj, resident);
  const int width = (int)ceil_div(nj, rounds);
  return rounds > 1 && !xcd_aligned(ni) && (int64_t)ni * width <= resident ? width : 0;
}

// Workgroups of a contraction whose row count, up to nj tiles of them, is on the device: those of
// the count that needs the most, for the splits it gets.  The most splits of the most tiles are
// mostly workgroups that exit, and a bound on the splits leaves few tiles without theirs.  16
// splits launched at most / this, grad_hidden and the step:
//    256 of 1024 rows, H = 2048, V = 131072   222 / 142 us   706 / 633 us  (32 splits of 8 tiles)
//    102 of 2048, H = 1024, V = 32000          34 /  22
//   1036 of 2048, H = 4096, V = 32000         454 / 232     1056 / 833
//   8212 recomputed, H = 3840, V = 262144                   51.6 / 51.2 ms
inline int counted_rows_grid(const GemmArgs& a, int tile) {
  int64_t grid = kXcds;
  for (int64_t j = 1; j <= a.nj; ++j) {
    const int64_t slab = j * tile * a.ldc;
    // (no count of j tiles takes more splits than the smallest)
    const int64_t rows = a.split_by_rows ? (j - 1) * tile + 1 : j * tile;
    const int ks = grad_hidden_k_splits(j * a.ni, a.max_splits, a.k_steps_plan, rows * a.ldc,
                                        resident_workgroups(tile));
    const int64_t held = std::max<int64_t>(1, a.slab_budget / slab);
    grid = std::max(grid, std::min<int64_t>(ks, held) * xcd_grid(j * a.ni));
  }
  return (int)grid;
}

template <class E, bool kAKMajor, bool kBKMajor>
int launch_gemm(GemmArgs a, int ksplit, int cls, hipStream_t stream) {
  static LdsOptIn lds;
  constexpr int kLdsBytes = kBKMajor ? E::kSmemBytes : kLaunchSmemBytes<E>;
  if (int rc = enable_large_lds(lce_gemm_nt_kernel<E, kAKMajor, kBKMajor>, kLdsBytes, lds))
    return rc;
  if (!kBKMajor && ksplit == 1 && a.m_dev == nullptr)
    a.j_chunk = round_chunk(a.ni, a.nj, E::kTile);
  const int ksteps = (int)ceil_div(a.k, E::kBK);
  a.k_per_split = (int)ceil_div(ksteps, ksplit) * E::kBK;
  // (with a device-side row count the kernel finds its number of splits itself)
  const bool counted = a.m_dev != nullptr && a.m_role == kRowsFollow;
  dim3 grid(counted ? counted_rows_grid(a, E::kTile)
            : a.j_chunk > 0 ? xcd_grid((int64_t)a.ni * a.j_chunk) * (int)ceil_div(a.nj, a.j_chunk)
                            : xcd_grid((int64_t)a.ni * a.nj), counted ? 1 : ksplit, 1);
  ScopedTimer timer(cls, stream);
  lce_gemm_nt_kernel<E, kAKMajor, kBKMajor><<<grid, E::kThreads, kLdsBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_transpose(const T* in, int64_t ld_in, int64_t rows, int64_t cols, T* out,
                     int64_t ld_out, int64_t out_cols, hipStream_t stream,
                     const int64_t* rows_dev = nullptr) {
  dim3 grid((unsigned)ceil_div(cols, 64), (unsigned)ceil_div(out_cols, 64), 1);
  TLCE_REQUIRE(grid.y <= 65535, "transpose: too many row tiles");
  ScopedTimer timer(kClassTranspose, stream);
  lce_transpose_pad_kernel<T><<<grid, 256, 0, stream>>>(in, ld_in, (int)rows, (int)cols, out,
                                                        ld_out, (int)out_cols, rows_dev);
  TLCE_LAUNCH_CHECK();
  return 0;
}

// Launchers of the engine-independent kernels (tlce_row_kernels.h), defined
// beside the C ABI.
int fill_zero(void* dst, int64_t bytes, hipStream_t stream);
int launch_k_tail(const void* matrix, int64_t rows, int64_t h, void* tail, hipStream_t stream);
// Copies of 16-bit weight [v, h] and hidden [m, h] (h a multiple of 8 but not of 64):
// weight_tail [v, 64] holds the columns after the last whole 64 and then zeros, hidden_copy
// [m, h rounded up to 64] the rows followed by zeros (of a row count on the device, m_dev, those).
int launch_column_tails(const void* weight, int64_t v, const void* hidden, int64_t m, int64_t h,
                        void* weight_tail, void* hidden_copy, const int64_t* m_dev,
                        hipStream_t stream);
int launch_token_scale(const ScaleArgs& sa, hipStream_t stream);
int launch_kl_finish(float* losses, const float* loss_part, const float* tsum_part, int n_tiles,
                     int64_t part_ld, const float* lse, int64_t m, hipStream_t stream);
int launch_topk_scan(const TopkScanArgs& sa, hipStream_t stream);
int launch_sum(const float* x, int64_t n, float* out, hipStream_t stream);

// ----------------------------------------------------------------- forward --
// Outputs of the vocabulary-shard forward (all null for the full-vocabulary one).
struct ShardStats {
  int64_t vocab_start = 0;
  float* local_max = nullptr;
  float* local_sum = nullptr;
  float* target_logits = nullptr;
};

// Merge of the forward's partials into lse, loss and (when asked for) the weighted loss sum;
// ca holds the operands, the partials and the plain outputs.  `weighted`: [m] scratch.
template <typename T>
int launch_combine(CombineArgs ca, int n_vtiles, int tile, int64_t m, const ShardStats& shard,
                   char* weighted, const RowOptions& opt, hipStream_t stream) {
  ca.label_offset = shard.vocab_start;
  ca.local_max = shard.local_max; ca.local_sum = shard.local_sum;
  ca.target_logits = shard.target_logits;
  ca.logit_scale = opt.logit_scale; ca.token_weights = opt.token_weights;
  ca.n_vtiles = n_vtiles; ca.tile = tile; ca.m_dev = opt.row_count;
  ca.weight_dim_first = opt.weight_dim_first;
  if (opt.weighted_sum != nullptr) {
    ca.weighted = reinterpret_cast<float*>(weighted);
    ca.weighted_rows = (int)m;
  }
  {
    ScopedTimer timer(kClassCombine, stream);
    lce_combine_loss_kernel<T><<<(int)ceil_div(m, kCombineRowsPerBlock),
                                64 * kCombineRowsPerBlock, 0, stream>>>(ca);
  }
  TLCE_LAUNCH_CHECK();
  if (opt.weighted_sum != nullptr) return launch_sum(ca.weighted, m, opt.weighted_sum, stream);
  return 0;
}

template <class E>
int forward_impl(const Plan& p, const void* hidden, const void* weight, const float* bias,
                 const int64_t* labels, const int64_t* row_idx, int64_t m, int64_t h, int64_t v,
                 int64_t ignore, int64_t exclude, float softcap, float* losses, float* lse,
                 float* valid_count, const ShardStats& shard, char* ws, hipStream_t stream,
                 const RowOptions& opt) {
  using T = typename E::T;
  const bool dynamic = opt.row_count != nullptr;
  const ForwardLayout l = forward_layout(p, dynamic, opt.weighted_sum != nullptr);
  ForwardArgs fa;
  fa.hidden = hidden; fa.weight = weight; fa.bias = bias;
  if (p.column_tail != 0) {
    char* hidden_copy = ws + l.tails + p.vp * 64 * 2;
    if (int rc = launch_column_tails(weight, v, hidden, m, h, ws + l.tails, hidden_copy,
                                     opt.row_count, stream))
      return rc;
    fa.weight_tail = ws + l.tails; fa.hidden = hidden_copy;
  }
  fa.m = (int)m; fa.h = (int)h; fa.v = (int)v;
  fa.exclude = exclude - shard.vocab_start; fa.softcap = softcap;
  fa.logit_scale = opt.logit_scale; fa.m_dev = opt.row_count;
  fa.n_ttiles = p.n_ttiles; fa.n_vtiles = p.n_vtiles; fa.nsplit = p.nsplit;
  fa.part_max = reinterpret_cast<float*>(ws + l.part_max);
  fa.part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  fa.part_ld = (int)p.mp;
  fa.kept = opt.kept;
  if (opt.weight_dim_first) {
    if (int rc = launch_forward_dim_first<E>(p, fa, stream)) return rc;
  } else {
    using Tail = typename ColumnTailOf<E>::type;
    if (int rc = p.column_tail != 0 ? launch_forward<Tail>(p, fa, stream)
                                    : launch_forward<E>(p, fa, stream))
      return rc;
  }

  CombineArgs ca;
  ca.hidden = hidden; ca.weight = weight; ca.bias = bias; ca.labels = labels;
  ca.row_idx = row_idx;
  ca.m = (int)m; ca.h = (int)h; ca.v = (int)v;
  ca.ignore = ignore; ca.exclude = exclude; ca.softcap = softcap;
  ca.part_max = fa.part_max; ca.part_sum = fa.part_sum;
  ca.part_ld = fa.part_ld; ca.nsplit = p.nsplit;
  ca.losses = losses; ca.lse = lse; ca.valid_count = valid_count;
  return launch_combine<T>(ca, p.n_vtiles, p.tile, m, shard, ws + l.weighted, opt, stream);
}

// ---------------------------------------------------------------- backward --
// The panel loop shared by every objective whose gradient is G . weight (and
// G^T . hidden): `produce(v0, width, g, gt)` fills the panel of rounded logit
// gradients for the vocabulary rows [v0, v0 + width); the loop contracts it
// into the float32 grad_hidden slabs and, when grad_weight != null, into the
// panel's rows of grad_weight, then casts / un-compacts grad_hidden.
template <class E, class Producer>
int panel_contractions(const Plan& p, const BackwardLayout& l, const void* hidden,
                       const void* weight, const int64_t* row_idx, int64_t m, int64_t n_out,
                       int64_t h, int64_t v, int dtype, void* grad_hidden, void* grad_weight,
                       char* ws, hipStream_t stream, Producer&& produce,
                       const std::function<int(float*)>& before_cast = nullptr,
                       const int64_t* m_dev = nullptr, bool dim_first = false) {
  using T = typename E::T;
  const bool weight_grad = grad_weight != nullptr;
  float* acc32 = reinterpret_cast<float*>(ws + l.acc32);
  T* wt = reinterpret_cast<T*>(ws + l.wt);
  T* ht = reinterpret_cast<T*>(ws + l.ht);
  T* g = reinterpret_cast<T*>(ws + l.g);
  T* gt = (weight_grad && !p.kmajor) ? reinterpret_cast<T*>(ws + l.gt) : nullptr;

  const T* hidden_t = static_cast<const T*>(hidden);
  const T* weight_t = static_cast<const T*>(weight);
  // the direct engine takes whole 64-row K slabs, the float32 engine any K
  constexpr int kSlab = sizeof(T) == 2 ? 64 : 1;
  const int64_t m64 = round_up(m, kSlab);
  if (!p.kmajor) {
    // K-contiguous copies for engines that cannot read K-major operands
    if (int rc = launch_transpose<T>(weight_t, h, v, h, wt, p.vp, p.vp, stream)) return rc;
    if (weight_grad) {
      if (int rc = launch_transpose<T>(hidden_t, h, m, h, ht, p.mp, p.mp, stream, m_dev))
        return rc;
    }
  } else {
    if (v % kSlab != 0) {
      if (int rc = launch_k_tail(weight_t, v, h, wt, stream)) return rc;
    }
    // (with a device-side row count the caller's buffer holds the padding rows)
    if (weight_grad && m_dev == nullptr && m % kSlab != 0) {
      if (int rc = launch_k_tail(hidden_t, m, h, ht, stream)) return rc;
    }
  }

  for (int panel = 0; panel < p.n_panels; ++panel) {
    const int64_t v0 = (int64_t)panel * p.vc;
    const int64_t width = std::min<int64_t>(p.vc, p.vp - v0);   // multiple of tile
    const int64_t rows_valid = std::min<int64_t>(p.vc, v - v0);  // real vocabulary rows
    if (int rc = produce(v0, width, g, gt)) return rc;

    GemmArgs dh;
    dh.b = g; dh.ldb = p.vc; dh.b_rows = (int)p.mp;
    dh.k_per_split = 0;
    dh.ni = p.n_htiles; dh.nj = p.n_ttiles;
    dh.c = acc32; dh.ldc = h; dh.c_rows = (int)m; dh.c_cols = (int)h;
    dh.c_split_stride = p.mp * h;
    dh.mode = (panel == 0) ? kStoreF32 : kAddF32;
    dh.m_dev = m_dev; dh.m_role = kRowsFollow;
    dh.slab_budget = p.dh_slab_rows * h;
    dh.max_splits = p.dh_max_ksplit;
    dh.k_steps_plan = (int)(p.vc / p.bk);
    GemmArgs dw;
    dw.m_dev = m_dev; dw.m_role = kKFollows; dw.m_round = p.bk;
    dw.k_per_split = 0;
    dw.ni = p.n_htiles; dw.nj = (int)(width / p.tile);
    dw.c = weight_grad ? static_cast<T*>(grad_weight) + v0 * h : nullptr; dw.ldc = h;
    dw.c_rows = (int)rows_valid; dw.c_cols = (int)h;
    dw.c_split_stride = 0;
    dw.mode = kStoreT;
    if constexpr (E::kHasKMajor) {
      if constexpr (kTakesDimFirst<E>) {
        if (dim_first) {
          // The head is stored [h, v].  grad_hidden: A = its columns [v0, v0+K), which
          // are K-contiguous rows of the stored matrix; B = G.
          dh.a = weight_t + v0; dh.lda = v; dh.a_rows = (int)h;
          dh.k = (int)round_up(rows_valid, kSlab);
          if (int rc = launch_gemm<E, false, false>(dh, p.dh_ksplit, kClassGradHidden, stream))
            return rc;
          if (weight_grad) {
            // grad_weight [h, v]: the roles of the operands swap so that the hidden axis
            // becomes the output's rows: A = G (its panel columns), B = hidden, both K-major
            GemmArgs dwt = dw;
            dwt.a = g; dwt.lda = p.vc; dwt.a_rows = (int)width;
            dwt.b = hidden_t; dwt.ldb = h; dwt.b_rows = (int)h;
            dwt.k = (int)m64;
            if (m64 != m && m_dev == nullptr) {
              dwt.b_tail = ht;
              dwt.b_k_full = (int)(m64 - kSlab);
            }
            dwt.ni = (int)(width / p.tile); dwt.nj = p.n_htiles;
            dwt.c = static_cast<T*>(grad_weight) + v0; dwt.ldc = v;
            dwt.c_rows = (int)h; dwt.c_cols = (int)rows_valid;
            if (int rc = launch_gemm<E, true, true>(dwt, 1, kClassGradWeight, stream)) return rc;
          }
          continue;
        }
      }
      if (p.kmajor) {
        // grad_hidden: A = weight rows [v0, v0+K) as stored (K-major), B = G
        dh.a = weight_t + v0 * h; dh.lda = h; dh.a_rows = (int)h;
        dh.k = (int)round_up(rows_valid, kSlab);
        if (dh.k != rows_valid) {
          dh.a_tail = wt;
          dh.a_k_full = dh.k - kSlab;
        }
        if (int rc = launch_gemm<E, true, false>(dh, p.dh_ksplit, kClassGradHidden, stream))
          return rc;
        if (weight_grad) {
          // grad_weight: A = hidden as stored, B = G as stored, both K-major (K = token)
          dw.a = hidden_t; dw.lda = h; dw.a_rows = (int)h;
          dw.b = g; dw.ldb = p.vc; dw.b_rows = (int)width;
          dw.k = (int)m64;
          if (m64 != m && m_dev == nullptr) {
            dw.a_tail = ht;
            dw.a_k_full = (int)(m64 - kSlab);
          }
          if (int rc = launch_gemm<E, true, true>(dw, 1, kClassGradWeight, stream)) return rc;
        }
        continue;
      }
    }
    dh.a = wt + v0; dh.lda = p.vp; dh.a_rows = (int)h;
    dh.k = (int)width;
    if (int rc = launch_gemm<E, false, false>(dh, p.dh_ksplit, kClassGradHidden, stream))
      return rc;
    if (weight_grad) {
      dw.a = ht; dw.lda = p.mp; dw.a_rows = (int)h;
      dw.b = gt; dw.ldb = p.mp; dw.b_rows = (int)width;
      dw.k = (int)p.mp;
      if (int rc = launch_gemm<E, false, false>(dw, 1, kClassGradWeight, stream)) return rc;
    }
  }

  if (before_cast) {
    if (int rc = before_cast(acc32)) return rc;   // extra float32 terms of grad_hidden
  }
  if (row_idx != nullptr || m_dev != nullptr) {
    if (int rc = fill_zero(grad_hidden, n_out * h * dtype_bytes(dtype), stream)) return rc;
  }
  {
    ScopedTimer timer(kClassOther, stream);
    lce_finalize_grad_hidden_kernel<T><<<(int)m, 256, 0, stream>>>(
        acc32, p.dh_ksplit, p.mp * h, p.dh_slab_rows * h, row_idx, (int)m, (int)h,
        static_cast<T*>(grad_hidden), m_dev, p.n_htiles, p.tile, p.dh_max_ksplit,
        (int)(p.vc / p.bk));
  }
  TLCE_LAUNCH_CHECK();
  return 0;
}

// vocab_start: global id of weight row 0 (labels and exclude are global ids).
// labels == null: the "gradient" panel holds softmax * probabilities_scale, so
// grad_hidden becomes the probability-weighted sum of weight rows.
template <class E>
int backward_impl(const Plan& p, const void* hidden, const void* weight, const float* bias,
                  const int64_t* labels, const int64_t* row_idx, const float* lse,
                  const float* valid_count, const float* grad_output, int64_t m, int64_t n_out,
                  int64_t h, int64_t v, int dtype, int reduction, int64_t ignore, int64_t exclude,
                  float softcap, int64_t vocab_start, void* grad_hidden, void* grad_weight,
                  float* grad_bias, char* ws, hipStream_t stream,
                  float probabilities_scale, const RowOptions& opt) {
  using T = typename E::T;
  const BackwardLayout l = backward_layout(p, m, h, dtype, grad_weight != nullptr);
  float* scale = reinterpret_cast<float*>(ws + l.scale);
  ScaleArgs sa;
  sa.labels = labels; sa.row_idx = row_idx; sa.grad_output = grad_output;
  sa.valid_count = valid_count; sa.m = (int)m; sa.mp = (int)p.mp; sa.reduction = reduction;
  sa.ignore = ignore; sa.scale = scale; sa.constant = probabilities_scale;
  // the gradient with respect to the raw dot products carries the logit multiplier
  sa.multiplier = opt.logit_scale;
  sa.token_weights = opt.token_weights; sa.m_dev = opt.row_count;
  if (int rc = launch_token_scale(sa, stream)) return rc;
  if (grad_bias != nullptr) {
    if (int rc = fill_zero(grad_bias, v * 4, stream)) return rc;
  }
  char* hidden_copy = ws + l.tails + p.vp * 64 * 2;   // p.column_tail
  if (p.column_tail != 0) {
    if (int rc = launch_column_tails(weight, v, hidden, m, h, ws + l.tails, hidden_copy,
                                     opt.row_count, stream))
      return rc;
  }
  auto produce = [&](int64_t v0, int64_t width, void* g, void* gt) -> int {
    GradLogitsArgs ga;
    ga.hidden = p.column_tail != 0 ? hidden_copy : hidden;
    ga.weight_tail = p.column_tail != 0 ? ws + l.tails : nullptr;
    ga.weight = weight; ga.bias = bias; ga.labels = labels;
    ga.lse = lse; ga.scale = scale;
    ga.m = (int)m; ga.h = (int)h; ga.v = (int)v;
    ga.ignore = ignore; ga.exclude = exclude - vocab_start; ga.softcap = softcap;
    ga.label_offset = vocab_start;
    ga.probabilities = (labels == nullptr) ? 1 : 0;
    ga.cap_grad = (labels == nullptr) ? 0 : 1;
    ga.logit_scale = opt.logit_scale; ga.m_dev = opt.row_count;
    ga.v0 = (int)v0;
    ga.n_ttiles = p.n_ttiles; ga.n_ptiles = (int)(width / p.tile);
    ga.g = g; ga.ldg = p.vc; ga.gt = gt; ga.ldgt = p.mp;
    ga.grad_bias = (bias != nullptr) ? grad_bias : nullptr;
    if constexpr (kKeepsLogits<E>) {
      const int kept = (int)std::min<int64_t>(ga.n_ptiles, opt.kept.v_tiles - v0 / p.tile);
      if (kept > 0) {   // the panel's first tiles
        GradLogitsArgs ka = ga;
        ka.n_ptiles = kept;
        if (int rc = launch_grad_from_kept<T>(ka, opt.kept, stream)) return rc;
        if (kept == ga.n_ptiles) return 0;
        ga.v0 += kept * p.tile;
        ga.n_ptiles -= kept;
        ga.g = static_cast<T*>(ga.g) + kept * p.tile;
      }
    }
    if (opt.weight_dim_first) return launch_grad_logits_dim_first<E>(ga, stream);
    using Tail = typename ColumnTailOf<E>::type;
    return p.column_tail != 0 ? launch_grad_logits<Tail>(ga, stream)
                              : launch_grad_logits<E>(ga, stream);
  };
  return panel_contractions<E>(p, l, hidden, weight, row_idx, m, n_out, h, v, dtype, grad_hidden,
                               grad_weight, ws, stream, produce, nullptr, opt.row_count,
                               opt.weight_dim_first);
}

// -------------------------------------------------------------- frozen KL ----
// KL(teacher || draft) of two frozen heads over one vocabulary
// (fused_dflash_kl_forward_cuda / _backward_cuda, fused_linear_ce_cuda.cu:1270-1509).
// Both heads run on one engine class (the less demanding of the two hidden sizes).
struct KlLayout {
  // stats: the teacher's forward partials, then the draft's per-tile partials
  // (part_max, part_sum, loss terms, teacher mass: n_vtiles x mp float32 each);
  // backward: BackwardLayout of the draft head
  int64_t stats, tile_part, ones, backward, total;
};

inline KlLayout kl_layout(const Plan& pd, const Plan& pt, int64_t m, int64_t hd, int dtype) {
  KlLayout l;
  l.stats = 0;
  l.tile_part = align256((int64_t)pd.n_vtiles * pd.mp * 4);
  int64_t off = std::max(4 * l.tile_part, forward_layout(pt).total);
  l.ones = off;      off += align256(pd.mp * 4);
  l.backward = off;  off += backward_layout(pd, m, hd, dtype, false).total;
  l.total = off;
  return l;
}

template <class E, bool kSoftcap, bool kGrad>
int launch_kl_panel_variant(const KlPanelArgs& a, hipStream_t stream) {
  static LdsOptIn lds;
  if (int rc = enable_large_lds(lce_kl_panel_kernel<E, kSoftcap, kGrad>, E::kSmemBytes, lds))
    return rc;
  const int grid = xcd_grid((int64_t)a.n_ttiles * a.n_ptiles);
  ScopedTimer timer(kClassGradLogits, stream);
  lce_kl_panel_kernel<E, kSoftcap, kGrad><<<grid, E::kThreads, E::kSmemBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

template <class E>
int launch_kl_panel(const KlPanelArgs& a, hipStream_t stream) {
  const bool grad = a.mode == kKlGrad;
  if (a.softcap > 0.0f) {
    return grad ? launch_kl_panel_variant<E, true, true>(a, stream)
                : launch_kl_panel_variant<E, true, false>(a, stream);
  }
  return grad ? launch_kl_panel_variant<E, false, true>(a, stream)
              : launch_kl_panel_variant<E, false, false>(a, stream);
}

// Teacher probabilities of the panel [v0, v0 + width), then the draft pass over it.
template <class E>
int kl_panel(const Plan& pd, const void* draft_hidden, const void* draft_weight,
             const void* teacher_hidden, const void* teacher_weight, const float* draft_lse,
             const float* teacher_lse, const float* ones, const float* scale, int64_t m,
             int64_t hd, int64_t ht, int64_t v, float softcap, int64_t v0, int64_t width,
             void* g, float* loss_part, float* tsum_part, float* part_max, float* part_sum,
             int mode, hipStream_t stream, void* kept = nullptr, int64_t kept_ld = 0,
             bool kept_is_written = false) {
  // kept: a buffer over the whole vocabulary [mp, kept_ld] that holds the teacher
  // probabilities between forward and backward.  The forward produces each panel into
  // it (and reads it there); the backward (kept_is_written) skips the producer and
  // reads the panel from it, writing the logit gradients to g.
  void* teacher_panel = kept != nullptr ? static_cast<char*>(kept) + v0 * (int64_t)sizeof(typename E::T) : g;
  const int64_t teacher_ld = kept != nullptr ? kept_ld : pd.vc;
  KlPanelArgs ka;
  ka.hidden = draft_hidden; ka.weight = draft_weight; ka.lse = draft_lse; ka.scale = scale;
  ka.m = (int)m; ka.h = (int)hd; ka.v = (int)v; ka.softcap = softcap;
  ka.v0 = (int)v0; ka.n_ttiles = pd.n_ttiles; ka.n_ptiles = (int)(width / pd.tile);
  ka.loss_part = loss_part; ka.tsum_part = tsum_part;
  ka.part_max = part_max; ka.part_sum = part_sum; ka.part_ld = (int)pd.mp; ka.mode = mode;
  if (kept != nullptr && kept_is_written) {
    ka.panel = g; ka.ld = pd.vc; ka.panel_in = teacher_panel; ka.ld_in = teacher_ld;
    return launch_kl_panel<E>(ka, stream);
  }
  GradLogitsArgs ga;
  ga.hidden = teacher_hidden; ga.weight = teacher_weight; ga.bias = nullptr;
  ga.labels = nullptr; ga.lse = teacher_lse; ga.scale = ones;
  ga.m = (int)m; ga.h = (int)ht; ga.v = (int)v;
  ga.ignore = 0; ga.exclude = -1; ga.softcap = softcap;
  ga.label_offset = 0; ga.probabilities = 1; ga.cap_grad = 0; ga.logit_scale = 1.0f;
  ga.v0 = (int)v0;
  ga.n_ttiles = pd.n_ttiles; ga.n_ptiles = (int)(width / pd.tile);
  ga.g = teacher_panel; ga.ldg = teacher_ld; ga.gt = nullptr; ga.ldgt = 0;
  ga.grad_bias = nullptr;
  if (int rc = launch_grad_logits<E>(ga, stream)) return rc;
  ka.panel = teacher_panel; ka.ld = teacher_ld;
  return launch_kl_panel<E>(ka, stream);
}

template <class E>
int kl_forward_impl(const Plan& pd, const Plan& pt, const KlLayout& l, const void* draft_hidden,
                    const void* draft_weight, const void* teacher_hidden,
                    const void* teacher_weight, int64_t m, int64_t hd, int64_t ht, int64_t v,
                    int dtype, float softcap, float* losses, float* draft_lse, float* teacher_lse,
                    char* ws, hipStream_t stream, void* kept_teacher = nullptr) {
  using T = typename E::T;
  // teacher statistics first: its probabilities need the teacher lse
  if (int rc = forward_impl<E>(pt, teacher_hidden, teacher_weight, nullptr, nullptr, nullptr, m,
                               ht, v, 0, -1, softcap, nullptr, teacher_lse, nullptr, ShardStats{},
                               ws + l.stats, stream, RowOptions{}))
    return rc;
  float* ones = reinterpret_cast<float*>(ws + l.ones);
  float* part_max = reinterpret_cast<float*>(ws + l.stats);
  float* part_sum = reinterpret_cast<float*>(ws + l.stats + l.tile_part);
  float* loss_part = reinterpret_cast<float*>(ws + l.stats + 2 * l.tile_part);
  float* tsum_part = reinterpret_cast<float*>(ws + l.stats + 3 * l.tile_part);
  ScaleArgs sa;
  sa.labels = nullptr; sa.row_idx = nullptr; sa.grad_output = nullptr; sa.valid_count = nullptr;
  sa.m = (int)m; sa.mp = (int)pd.mp; sa.reduction = TLCE_REDUCTION_SUM; sa.ignore = 0;
  sa.scale = ones; sa.constant = 1.0f; sa.multiplier = 1.0f;
  if (int rc = launch_token_scale(sa, stream)) return rc;
  // one pass over the draft head per panel: loss terms and the draft's per-tile
  // softmax partials (the teacher partials above are dead by now)
  const BackwardLayout bl = backward_layout(pd, m, hd, dtype, false);
  void* g = ws + l.backward + bl.g;
  // teacher probabilities that go to a buffer over the whole vocabulary need no bounded
  // panel: one launch of each kernel covers all of it (fewer partly filled last rounds)
  const int n_panels = kept_teacher != nullptr ? 1 : pd.n_panels;
  const int64_t panel_width = kept_teacher != nullptr ? pd.vp : pd.vc;
  for (int panel = 0; panel < n_panels; ++panel) {
    const int64_t v0 = (int64_t)panel * panel_width;
    const int64_t width = std::min<int64_t>(panel_width, pd.vp - v0);
    if (int rc = kl_panel<E>(pd, draft_hidden, draft_weight, teacher_hidden, teacher_weight,
                             nullptr, teacher_lse, ones, nullptr, m, hd, ht, v, softcap, v0,
                             width, g, loss_part, tsum_part, part_max, part_sum, kKlLoss,
                             stream, kept_teacher, pd.vp, false))
      return rc;
  }
  CombineArgs ca;
  ca.hidden = draft_hidden; ca.weight = draft_weight; ca.bias = nullptr; ca.labels = nullptr;
  ca.row_idx = nullptr;
  ca.m = (int)m; ca.h = (int)hd; ca.v = (int)v;
  ca.ignore = 0; ca.exclude = -1; ca.softcap = softcap;
  ca.part_max = part_max; ca.part_sum = part_sum;
  ca.part_ld = (int)pd.mp; ca.nsplit = pd.n_vtiles;
  ca.losses = nullptr; ca.lse = draft_lse; ca.valid_count = nullptr;
  ca.label_offset = 0; ca.local_max = nullptr; ca.local_sum = nullptr; ca.target_logits = nullptr;
  {
    ScopedTimer timer(kClassCombine, stream);
    lce_combine_loss_kernel<T><<<(int)ceil_div(m, kCombineRowsPerBlock),
                                64 * kCombineRowsPerBlock, 0, stream>>>(ca);
    TLCE_LAUNCH_CHECK();
    if (int rc = launch_kl_finish(losses, loss_part, tsum_part, pd.n_vtiles, pd.mp, draft_lse, m,
                                  stream))
      return rc;
  }
  return 0;
}

template <class E>
int kl_backward_impl(const Plan& pd, const KlLayout& l, const void* draft_hidden,
                     const void* draft_weight, const void* teacher_hidden,
                     const void* teacher_weight, const float* draft_lse, const float* teacher_lse,
                     const float* grad_output, int64_t m, int64_t hd, int64_t ht, int64_t v,
                     int dtype, float softcap, void* grad_hidden, char* ws, hipStream_t stream,
                     const void* kept_teacher = nullptr) {
  float* ones = reinterpret_cast<float*>(ws + l.ones);
  char* bws = ws + l.backward;
  const BackwardLayout bl = backward_layout(pd, m, hd, dtype, false);
  float* scale = reinterpret_cast<float*>(bws + bl.scale);
  ScaleArgs sa;
  sa.labels = nullptr; sa.row_idx = nullptr; sa.grad_output = nullptr; sa.valid_count = nullptr;
  sa.m = (int)m; sa.mp = (int)pd.mp; sa.reduction = TLCE_REDUCTION_NONE; sa.ignore = 0;
  sa.scale = ones; sa.constant = 1.0f; sa.multiplier = 1.0f;
  if (int rc = launch_token_scale(sa, stream)) return rc;
  sa.grad_output = grad_output; sa.scale = scale;   // scale[r] = grad_output[r]
  if (int rc = launch_token_scale(sa, stream)) return rc;
  auto produce = [&](int64_t v0, int64_t width, void* g, void*) -> int {
    return kl_panel<E>(pd, draft_hidden, draft_weight, teacher_hidden, teacher_weight, draft_lse,
                       teacher_lse, ones, scale, m, hd, ht, v, softcap, v0, width, g, nullptr,
                       nullptr, nullptr, nullptr, kKlGrad, stream,
                       const_cast<void*>(kept_teacher), pd.vp, kept_teacher != nullptr);
  };
  return panel_contractions<E>(pd, bl, draft_hidden, draft_weight, nullptr, m, m, hd, v, dtype,
                               grad_hidden, nullptr, bws, stream, produce);
}

// ------------------------------------------------ cross entropy + top-k ----
struct TopkPlan {
  Plan plan;            // engine, tiles and the backward's panels (input dtype)
  int64_t vcf;          // columns of a float32 logits panel
  int n_fpanels;
  int64_t run_max, run_sum, fpanel, forward_total;
  int64_t ce_scale, backward, backward_total;
};

inline TopkPlan topk_plan(int64_t m, int64_t h, int64_t v, int dtype, int64_t panel_bytes) {
  TopkPlan t;
  t.plan = make_plan(m, h, v, dtype, false, panel_bytes);
  const Plan& p = t.plan;
  if (panel_bytes <= 0) panel_bytes = kDefaultPanelBytes;
  int64_t tiles = std::max<int64_t>(1, panel_bytes / (p.mp * 4) / p.tile);
  tiles = std::min<int64_t>(tiles, p.n_vtiles);
  if (tiles >= 16 && tiles < p.n_vtiles) tiles = tiles / 16 * 16;
  t.vcf = tiles * p.tile;
  t.n_fpanels = (int)ceil_div(p.vp, t.vcf);
  int64_t off = 0;
  t.run_max = off;  off += align256(m * 4);
  t.run_sum = off;  off += align256(m * 4);
  t.fpanel = off;   off += align256(p.mp * t.vcf * 4);
  t.forward_total = off;
  off = 0;
  t.ce_scale = off; off += align256(p.mp * 4);
  t.backward = off; off += backward_layout(p, m, h, dtype, false).total;
  t.backward_total = off;
  return t;
}

template <class E, bool kSoftcap>
int launch_logits_panel_variant(const LogitsPanelArgs& a, hipStream_t stream) {
  static LdsOptIn lds;
  if (int rc = enable_large_lds(lce_logits_panel_kernel<E, kSoftcap>, E::kSmemBytes, lds))
    return rc;
  const int grid = xcd_grid((int64_t)a.n_ttiles * a.n_ptiles);
  ScopedTimer timer(kClassGradLogits, stream);
  lce_logits_panel_kernel<E, kSoftcap><<<grid, E::kThreads, E::kSmemBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

// After the scan of a float32 logits panel: exp(logit - the row's largest logit so
// far) * cap' of that panel, rounded to bf16, into a panel over the whole vocabulary
// (the operand of the gradient contraction formed in the forward).
struct ExpFromLogitsArgs {
  const float* logits;   // [m, ld] float32 (columns past the vocabulary hold -inf)
  int64_t ld;
  int m, m_pad;          // rows with logits; rows of `out` to define (zeros from m on)
  int width;             // columns of this logits panel, a multiple of 8
  float softcap;
  const float* run_max;  // [m] the reference: the row's largest logit so far
  float* ref_used;       // [m] out: the reference this panel was written with
  void* out;             // bf16 [m_pad, ld_out]; this panel goes to columns col0 ...
  int64_t ld_out, col0;
};
int launch_exp_from_logits(const ExpFromLogitsArgs& a, hipStream_t stream);

struct TopkExpHook {
  void* panel;           // bf16 [m_pad, ld]
  int64_t ld;
  int m_pad;
  float* ref_used;       // [n_fpanels, m_pad]
};

template <class E>
int topk_forward_impl(const TopkPlan& t, const void* hidden, const void* weight,
                      const int64_t* labels, int64_t m, int64_t h, int64_t v, int top_k,
                      float multiplier, float softcap, float* losses, float* probabilities,
                      float* top_values, int64_t* top_ids, float* lse, char* ws,
                      hipStream_t stream, const TopkExpHook* hook = nullptr,
                      const int* run_flag = nullptr) {
  // run_flag: only the lists, and only if *run_flag != 0 (losses, probabilities and lse
  // have been written from another pass over the logits)
  using T = typename E::T;
  const Plan& p = t.plan;
  float* run_max = reinterpret_cast<float*>(ws + t.run_max);
  float* run_sum = reinterpret_cast<float*>(ws + t.run_sum);
  float* panel = reinterpret_cast<float*>(ws + t.fpanel);
  for (int pi = 0; pi < t.n_fpanels; ++pi) {
    const int64_t v0 = (int64_t)pi * t.vcf;
    const int64_t width = std::min<int64_t>(t.vcf, p.vp - v0);
    const int64_t valid = std::min<int64_t>(t.vcf, v - v0);
    LogitsPanelArgs la;
    la.hidden = hidden; la.weight = weight;
    la.m = (int)m; la.h = (int)h; la.v = (int)v;
    la.softcap = softcap; la.logit_scale = multiplier;
    la.v0 = (int)v0; la.n_ttiles = p.n_ttiles; la.n_ptiles = (int)(width / p.tile);
    la.panel = panel; la.ld = t.vcf; la.run_flag = run_flag;
    if (softcap > 0.0f) {
      if (int rc = launch_logits_panel_variant<E, true>(la, stream)) return rc;
    } else {
      if (int rc = launch_logits_panel_variant<E, false>(la, stream)) return rc;
    }
    TopkScanArgs sa;
    sa.panel = panel; sa.ld = t.vcf; sa.m = (int)m; sa.v0 = v0; sa.width = (int)valid;
    sa.stored = (int)width; sa.k = top_k; sa.first = pi == 0;
    sa.run_max = run_max; sa.run_sum = run_sum; sa.top_values = top_values; sa.top_ids = top_ids;
    sa.run_flag = run_flag;
    if (int rc = launch_topk_scan(sa, stream)) return rc;
    if (hook != nullptr) {
      ExpFromLogitsArgs xa;
      xa.logits = panel; xa.ld = t.vcf; xa.m = (int)m; xa.m_pad = hook->m_pad;
      xa.width = (int)width; xa.softcap = softcap;
      xa.run_max = run_max; xa.ref_used = hook->ref_used + (int64_t)pi * hook->m_pad;
      xa.out = hook->panel; xa.ld_out = hook->ld; xa.col0 = v0;
      if (int rc = launch_exp_from_logits(xa, stream)) return rc;
    }
  }
  if (run_flag != nullptr) return 0;
  TopkFinishArgs fa;
  fa.hidden = hidden; fa.weight = weight; fa.labels = labels; fa.m = (int)m; fa.h = (int)h;
  fa.softcap = softcap; fa.logit_scale = multiplier;
  fa.run_max = run_max; fa.run_sum = run_sum;
  fa.lse = lse; fa.losses = losses; fa.probabilities = probabilities;
  {
    ScopedTimer timer(kClassCombine, stream);
    lce_topk_finish_kernel<T><<<(int)ceil_div(m, 4), 256, 0, stream>>>(fa);
  }
  TLCE_LAUNCH_CHECK();
  return 0;
}

template <class E>
int topk_backward_impl(const TopkPlan& t, const void* hidden, const void* weight,
                       const int64_t* labels, const float* lse, const int64_t* top_ids,
                       const float* ce_scale, const float* grad_top_values, int64_t m, int64_t h,
                       int64_t v, int dtype, int top_k, float multiplier, float softcap,
                       void* grad_hidden, char* ws, hipStream_t stream) {
  using T = typename E::T;
  const Plan& p = t.plan;
  char* bws = ws + t.backward;
  const BackwardLayout bl = backward_layout(p, m, h, dtype, false);
  float* scale = reinterpret_cast<float*>(bws + bl.scale);
  // scale[r] = ce_scale[r] * multiplier: d loss / d raw logit carries the multiplier
  ScaleArgs sa;
  sa.labels = nullptr; sa.row_idx = nullptr; sa.grad_output = ce_scale; sa.valid_count = nullptr;
  sa.m = (int)m; sa.mp = (int)p.mp; sa.reduction = TLCE_REDUCTION_NONE; sa.ignore = 0;
  sa.scale = scale; sa.constant = 0.0f; sa.multiplier = multiplier;
  if (int rc = launch_token_scale(sa, stream)) return rc;
  auto produce = [&](int64_t v0, int64_t width, void* g, void* gt) -> int {
    GradLogitsArgs ga;
    ga.hidden = hidden; ga.weight = weight; ga.bias = nullptr; ga.labels = nullptr;
    ga.lse = lse; ga.scale = scale;
    ga.m = (int)m; ga.h = (int)h; ga.v = (int)v;
    ga.ignore = 0; ga.exclude = -1; ga.softcap = softcap;
    ga.label_offset = 0; ga.probabilities = 1; ga.cap_grad = 1; ga.logit_scale = multiplier;
    ga.v0 = (int)v0;
    ga.n_ttiles = p.n_ttiles; ga.n_ptiles = (int)(width / p.tile);
    ga.g = g; ga.ldg = p.vc; ga.gt = gt; ga.ldgt = p.mp;
    ga.grad_bias = nullptr;
    return launch_grad_logits<E>(ga, stream);
  };
  auto single_rows = [&](float* acc32) -> int {
    // with a K split the label / top-k terms go to the first slab only
    TopkAdjustArgs aa;
    aa.hidden = hidden; aa.weight = weight; aa.labels = labels; aa.top_ids = top_ids;
    aa.ce_scale = ce_scale; aa.grad_top_values = grad_top_values;
    aa.m = (int)m; aa.h = (int)h; aa.v = (int)v; aa.k = top_k;
    aa.softcap = softcap; aa.logit_scale = multiplier; aa.acc32 = acc32;
    ScopedTimer timer(kClassOther, stream);
    lce_topk_adjust_kernel<T><<<(int)m, 256, 0, stream>>>(aa);
    TLCE_LAUNCH_CHECK();
    return 0;
  };
  return panel_contractions<E>(p, bl, hidden, weight, nullptr, m, m, h, v, dtype, grad_hidden,
                               nullptr, bws, stream, produce, single_rows);
}



struct SoftEmbeddingLayout {
  int64_t forward_ws, lse, backward_ws, total;
};

inline SoftEmbeddingLayout soft_embedding_layout(const Plan& fp, const Plan& bp, int64_t m, int64_t h,
                                          int dtype) {
  SoftEmbeddingLayout l;
  l.forward_ws = 0;
  l.lse = round_up(forward_layout(fp).total, 256);
  l.backward_ws = l.lse + round_up(m * 4, 256);
  l.total = l.backward_ws + backward_layout(bp, m, h, dtype, false).total;
  return l;
}

template <class E>
int soft_embedding_impl(const Plan& fp, const Plan& bp, const SoftEmbeddingLayout& l,
                        const void* hidden, const void* weight, int64_t m, int64_t h, int64_t v,
                        int dtype, float softcap, float scale, void* out, char* ws,
                        hipStream_t stream) {
  float* lse = reinterpret_cast<float*>(ws + l.lse);
  if (int rc = forward_impl<E>(fp, hidden, weight, nullptr, nullptr, nullptr, m, h, v, 0, -1,
                               softcap, nullptr, lse, nullptr, ShardStats{}, ws + l.forward_ws,
                               stream, RowOptions{}))
    return rc;
  return backward_impl<E>(bp, hidden, weight, nullptr, nullptr, nullptr, lse, nullptr, nullptr, m,
                          m, h, v, dtype, TLCE_REDUCTION_SUM, 0, -1, softcap, 0, out, nullptr,
                          nullptr, ws + l.backward_ws, stream, scale, RowOptions{});
}


// The kernel launchers of one engine, by kernel family.  An engine whose
// kernels compile slowly is built as several translation units, one family
// each; X is `template` in the unit that owns the family and `extern template`
// in the others.
#define TLCE_LAUNCHERS_FORWARD(X, E) \
  X int launch_forward<E>(const Plan&, const ForwardArgs&, hipStream_t);
#define TLCE_LAUNCHERS_GRAD_LOGITS(X, E, kSoftcap, kBias) \
  X int launch_grad_logits_variant<E, kSoftcap, kBias>(const GradLogitsArgs&, hipStream_t);
#define TLCE_LAUNCHERS_FORWARD_DIM_FIRST(X, E) \
  X int launch_forward_dim_first<E>(const Plan&, const ForwardArgs&, hipStream_t);
#define TLCE_LAUNCHERS_GRAD_LOGITS_DIM_FIRST(X, E) \
  X int launch_grad_logits_dim_first<E>(const GradLogitsArgs&, hipStream_t);
#define TLCE_LAUNCHERS_GEMM(X, E)                                         \
  X int launch_gemm<E, false, false>(GemmArgs, int, int, hipStream_t);    \
  X int launch_gemm<E, true, false>(GemmArgs, int, int, hipStream_t);     \
  X int launch_gemm<E, true, true>(GemmArgs, int, int, hipStream_t);
#define TLCE_LAUNCHERS_KL(X, E) \
  X int launch_kl_panel<E>(const KlPanelArgs&, hipStream_t);
#define TLCE_LAUNCHERS_LOGITS(X, E)                                                     \
  X int launch_logits_panel_variant<E, true>(const LogitsPanelArgs&, hipStream_t);      \
  X int launch_logits_panel_variant<E, false>(const LogitsPanelArgs&, hipStream_t);

// The per-engine launch sequences the C ABI dispatches to.  X is `extern
// template` where they are used and `template` in the translation unit that
// instantiates engine E.
#define TLCE_ENGINE_ENTRY_POINTS(X, E)                                                          \
  X int forward_impl<E>(const Plan&, const void*, const void*, const float*, const int64_t*,    \
                        const int64_t*, int64_t, int64_t, int64_t, int64_t, int64_t, float,     \
                        float*, float*, float*, const ShardStats&, char*, hipStream_t,          \
                        const RowOptions&);                                                     \
  X int backward_impl<E>(const Plan&, const void*, const void*, const float*, const int64_t*,   \
                         const int64_t*, const float*, const float*, const float*, int64_t,     \
                         int64_t, int64_t, int64_t, int, int, int64_t, int64_t, float, int64_t, \
                         void*, void*, float*, char*, hipStream_t, float, const RowOptions&);   \
  X int soft_embedding_impl<E>(const Plan&, const Plan&, const SoftEmbeddingLayout&,            \
                               const void*, const void*, int64_t, int64_t, int64_t, int, float, \
                               float, void*, char*, hipStream_t);                               \
  X int kl_forward_impl<E>(const Plan&, const Plan&, const KlLayout&, const void*, const void*, \
                           const void*, const void*, int64_t, int64_t, int64_t, int64_t, int,   \
                           float, float*, float*, float*, char*, hipStream_t, void*);           \
  X int kl_backward_impl<E>(const Plan&, const KlLayout&, const void*, const void*,             \
                            const void*, const void*, const float*, const float*, const float*, \
                            int64_t, int64_t, int64_t, int64_t, int, float, void*, char*,       \
                            hipStream_t, const void*);                                          \
  X int topk_forward_impl<E>(const TopkPlan&, const void*, const void*, const int64_t*,         \
                             int64_t, int64_t, int64_t, int, float, float, float*, float*,      \
                             float*, int64_t*, float*, char*, hipStream_t,                      \
                             const TopkExpHook*, const int*);                                   \
  X int topk_backward_impl<E>(const TopkPlan&, const void*, const void*, const int64_t*,        \
                              const float*, const int64_t*, const float*, const float*,         \
                              int64_t, int64_t, int64_t, int, int, float, float, void*, char*,  \
                              hipStream_t);

}  // namespace tlce
