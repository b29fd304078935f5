// Forward that also leaves the gradients: three contractions instead of four.
//
// The plain forward keeps no logits, so the backward has to recompute them
// (ce_grad_logits_kernel works on stored logits, fused_linear_ce_cuda.cu:240-290;
// the reference's blocks hold float32 logits between its forward and backward
// halves, :618-791).  When the loss is reduced to a scalar ("mean" / "sum") the
// upstream gradient is one number, and the gradients of the loss SUM can be
// formed while the logits of a block of rows exist, then scaled by that number
// afterwards.  Rows are taken in blocks of as many rows as a bounded panel holds
// over the WHOLE vocabulary; per block:
//
//   1. lce_exp_logits_panel_kernel: one contraction; the panel receives
//      e[r, v] = exp(z[r, v] - c[r]) * cap'(z) rounded to bf16, where
//      c[r] is a per-row reference logit known beforehand (the label's logit, a
//      one-row dot product).  Any c within ~80 of the row maximum keeps e inside
//      bf16's exponent range (float32's) with full relative precision.  The
//      tile sums of exp(z - c) and the tile maxima go out as per-tile partials.
//   2. lce_fused_rows_kernel: lse[r] = c[r] + log(sum), loss, the row factor
//      s[r] = weight[r] / sum (softmax = s * e), the label's panel entry replaced
//      by (e_label - sum) * cap' so that s * entry = (p_label - 1) * cap', and
//      hidden rows scaled by s for the grad_weight contraction.  A row whose
//      maximum lies outside [c - 40, c + 40] marks the block; steps 1-2 are
//      launched a second time and run only for marked blocks, with c = the exact
//      row maximum found by the first try (cannot fail again).
//   3. grad_hidden[r, :] = s[r] * (panel . weight)[r, :]   (K = the vocabulary,
//      complete for the block: no read-modify-write of a slab across panels)
//   4. grad_weight += panel^T . (s * hidden)   (float32 accumulator [v, h], one
//      read-modify-write per block of rows)
//
// Both gradients stay float32 until the upstream gradient arrives
// (lce_scale_cast_rows_kernel), so each is rounded once.
#pragma once

#include "tlce_host.h"
#include "tlce_split_f32.h"

namespace tlce {

// The row offset beyond which the first try is redone with the exact maximum
// (natural-log units).  exp(40) ~ 2e17 and its reciprocal are far inside the
// bf16 / float32 exponent range, also after a multiplication by a hidden entry
// or a loss weight.  f16 (largest number 65504) has no such room: the label's
// panel entry alone is of the size of sum_v exp(z - c) = 1 / softmax(label), so
// the sequence is built for bf16 only and f16 inputs keep the recomputing backward.
// Default bound of the panel of exponentiated logits: 32 token tiles over a
// 152 K vocabulary in 16-bit.  Per block of rows the grad_weight accumulator
// [v, h] float32 is read and written once, so fewer, larger blocks cost less
// (measured at 32768 x 4096 x 151936: 1 GiB 106.7 ms per step, 1.2 GiB 101.5,
// 2.4 GiB 96.9).
constexpr int64_t kDefaultFusedPanelBytes = 5ll << 29;
constexpr float kRefWindow = 40.0f;

struct ExpPanelArgs {
  const void* hidden;   // [m, h] the rows of this block
  const void* weight;   // [v, h]
  const float* ref;     // [m] reference logit per row (natural units); +inf: row without loss
  float ref_const = 0.0f;   // ref == null: the reference of every row
  int m, h, v;
  int64_t exclude;
  float softcap;
  float logit_scale;    // logits = cap(logit_scale * hidden . weight^T)
  int n_ttiles, n_vtiles;
  void* panel;          // [n_ttiles * tile, ld]
  int64_t ld;
  float* part_sum;      // [n_vtiles, part_ld] sum over the tile of exp(z - ref)
  float* part_max;      // [n_vtiles, part_ld] tile maximum of z in base-2 units
  int part_ld;
  const int* run_flag;  // non-null: the launch does nothing unless *run_flag != 0
  float* part_entry = nullptr;     // [n_vtiles, part_ld] sum over the tile of the entries,
  float* part_rounded = nullptr;   // exact and rounded (kRounded)
  // Row count known only to the device (null: m is exact): m is then the block's
  // capacity, and the block holds rows [row0, row0 + m) of the counted rows.
  const int64_t* m_dev = nullptr;
  int64_t row0 = 0;
  bool tail_last = false;   // the tiles of a narrow last row of tiles come after all others
};

// kPlain: the panel receives exp(z - c) itself, without the soft cap's derivative
// (a forward value, the unnormalised softmax, not a logit gradient).
// kRounded: the sums of the entries before and after their rounding go out as well, so that
// the factor common to a row's rounding errors can be taken out again.
// One tile of the panel; a narrow engine's holds fewer tokens.
template <class E, bool kSoftcap, bool kPlain, bool kRounded>
__device__ __forceinline__ void exp_logits_tile(ExpPanelArgs p, int tt, int vt, char* smem) {
  using T = typename E::T;
  E eng;
  typename E::Acc acc;
  const int vbase = vt * E::kTile;
  // Reference logit of every token column of the tile in base-2 units; +inf for
  // rows past the block and rows without loss, whose whole column of e becomes 0.
  // Fetched before the contraction so that the latency passes under it, and parked
  // in the LDS beyond the engine's stages: during the main loop every register
  // of the wave is taken.
  float* ref_stash = reinterpret_cast<float*>(smem + E::kSmemBytes);
  for (int c = threadIdx.x; c < E::kTile; c += E::kThreads) {
    const int r = tt * E::kTile + c;
    ref_stash[c] = (r < p.m) ? (p.ref != nullptr ? p.ref[r] : p.ref_const) * TLCE_LOG2E
                             : INFINITY;
  }
  eng.mainloop_set(static_cast<const T*>(p.weight), p.h, vbase, p.v,
                   static_cast<const T*>(p.hidden), p.h, tt * E::kTile, p.m, 0, p.h, acc, smem);
  // (the main loop's barriers have made the stash visible to every wave)
  float ref2[E::kCols];
#pragma unroll
  for (int j = 0; j < E::kCols; ++j) ref2[j] = ref_stash[eng.col(j)];

  const float inv_cap = kSoftcap ? p.logit_scale / p.softcap : 0.0f;
  const float to_base2 = kSoftcap ? p.softcap * TLCE_LOG2E : p.logit_scale * TLCE_LOG2E;
  const bool edge = (vbase + E::kTile > p.v) ||
                    (p.exclude >= vbase && p.exclude < vbase + E::kTile);
  const int excluded = (int)p.exclude;
  float col_sum[E::kCols], col_max[E::kCols];
  float col_entry[kRounded ? E::kCols : 1], col_rounded[kRounded ? E::kCols : 1];
  T* panel = static_cast<T*>(p.panel);
  const int pcol = vt * E::kTile;   // first panel column of this tile

  // The tile is staged in LDS (free after the main loop) as [token][vocab]:
  // 512-byte rows, 16-byte chunk c of token t in slot c ^ (t & 31), and leaves in
  // whole rows, a quarter of the tokens (one owned column index) at a time.  Entries in
  // three planes ([token][plane][vocab]) take 96 KiB a quarter, each in the same place.
  constexpr int kQuarter = E::kStageCols * E::kTokensPerIndex;   // tokens
  constexpr int kPlaneBytes = kQuarter * 512;
  auto emit = [&](auto edge_tag) {
    constexpr bool kEdge = decltype(edge_tag)::value;
    asm volatile("" ::: "memory");   // one real branch per variant
#pragma unroll
    for (int j = 0; j < E::kCols; ++j) {
      const int tok = E::kPlanes > 1
                          ? (j % E::kStageCols) * E::kTokensPerIndex + eng.position_in_index()
                          : eng.col(j);
      float s = 0.0f, mx = -INFINITY, entry = 0.0f, rounded = 0.0f;
#pragma unroll
      for (int i = 0; i < E::kRows; i += 4) {
        float e4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = eng.row(i + q);
          float z2, dcap = 1.0f;
          if (kSoftcap) {
            const float t = tanh_of<E::kPrecise>(element_of<E>(acc, j, i + q) * inv_cap);
            z2 = t * to_base2;
            dcap = 1.0f - t * t;
          } else {
            z2 = element_of<E>(acc, j, i + q) * to_base2;
          }
          float e = exp2_of<E::kPrecise>(z2 - ref2[j]);
          if (kEdge) {
            const bool ok = (vbase + row < p.v) && (vbase + row != excluded);
            e = ok ? e : 0.0f;
            z2 = ok ? z2 : -INFINITY;
          }
          mx = fmaxf(mx, z2);
          s += e;
          e4[q] = (kSoftcap && !kPlain) ? e * dcap : e;
        }
        const int vq = eng.row(i) >> 2;
        char* dst = smem + tok * 512 + (((vq >> 1) ^ (tok & 31)) * 16) + (vq & 1) * 8;
        if constexpr (E::kPlanes > 1) {
          float part[4][3];
#pragma unroll
          for (int q = 0; q < 4; ++q) split_planes(e4[q], part[q]);
#pragma unroll
          for (int pl = 0; pl < 3; ++pl)
            store4<T>(reinterpret_cast<T*>(dst + pl * kPlaneBytes), part[0][pl], part[1][pl],
                      part[2][pl], part[3][pl]);
        } else {
          store4<T>(reinterpret_cast<T*>(dst), e4[0], e4[1], e4[2], e4[3]);
          if (kRounded) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (kSoftcap) entry += e4[q];
              rounded += to_float<T>(from_float<T>(e4[q]));
            }
          }
        }
        // summed here: left to the compiler the sums of a column move to where they are used,
        // and the entries wait for them in scratch memory
        asm volatile("" : "+v"(s), "+v"(mx));
      }
      col_sum[j] = s;
      col_max[j] = mx;
      if (kRounded) {
        col_entry[j] = kSoftcap ? entry : s;
        col_rounded[j] = rounded;
      }
      if (E::kReadsWhereUsed) __builtin_amdgcn_sched_barrier(0);
      if (j % E::kStageCols != E::kStageCols - 1) continue;
      __syncthreads();
      if constexpr (E::kPlanes > 1) {
#pragma unroll 4
        for (int it = 0; it < 3 * kQuarter * 32 / E::kThreads; ++it) {
          const int c = it * E::kThreads + threadIdx.x;
          const int pl = c / (kQuarter * 32), sl = (c % (kQuarter * 32)) >> 5, ch = c & 31;
          const int t = E::token_of_index(j + 1 - E::kStageCols + sl / E::kTokensPerIndex,
                                          sl % E::kTokensPerIndex);
          const uint4 val = *reinterpret_cast<const uint4*>(smem + pl * kPlaneBytes + sl * 512 +
                                                            ((ch ^ (sl & 31)) * 16));
          stream_store16(panel + (((int64_t)tt * E::kTile + t) * 3 + pl) * p.ld + pcol + ch * 8,
                         val);
        }
        if (j + 1 < E::kCols) __syncthreads();   // the quarter has been read out
        continue;
      }
      constexpr int kPieces = E::kTokensPerIndex * 32;   // 16-byte pieces per owned index
#pragma unroll
      for (int it = 0; it < E::kStageCols * kPieces / E::kThreads; ++it) {
        const int c = it * E::kThreads + threadIdx.x;
        const int t = E::token_of_index(j + 1 - E::kStageCols + c / kPieces, (c % kPieces) >> 5);
        const int ch = c & 31;
        const uint4 val = *reinterpret_cast<const uint4*>(smem + t * 512 + ((ch ^ (t & 31)) * 16));
        stream_store16(panel + ((int64_t)tt * E::kTile + t) * p.ld + pcol + ch * 8, val);
      }
    }
  };
  if (edge) {
    emit(std::true_type{});
  } else {
    emit(std::false_type{});
  }

  // merge the kShare threads that hold the same token column, in a fixed order
  __syncthreads();   // the last quarter has been read out of the stage
  float* sh_sum = reinterpret_cast<float*>(smem);
  float* sh_max = sh_sum + E::kShare * E::kTile;
  const int slot = eng.share_slot();
#pragma unroll
  for (int j = 0; j < E::kCols; ++j) {
    sh_sum[slot * E::kTile + eng.col(j)] = col_sum[j];
    sh_max[slot * E::kTile + eng.col(j)] = col_max[j];
  }
  __syncthreads();
  for (int c = threadIdx.x; c < E::kTileB; c += E::kThreads) {
    float sum = 0.0f, mx = -INFINITY;
#pragma unroll
    for (int sl = 0; sl < E::kShare; ++sl) {
      sum += sh_sum[sl * E::kTile + c];
      mx = fmaxf(mx, sh_max[sl * E::kTile + c]);
    }
    const int64_t o = (int64_t)vt * p.part_ld + tt * E::kTile + c;
    p.part_sum[o] = sum;
    p.part_max[o] = mx;
  }
  if (kRounded) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E::kCols; ++j) {
      sh_sum[slot * E::kTile + eng.col(j)] = col_entry[j];
      sh_max[slot * E::kTile + eng.col(j)] = col_rounded[j];
    }
    __syncthreads();
    for (int c = threadIdx.x; c < E::kTileB; c += E::kThreads) {
      float entry = 0.0f, rounded = 0.0f;
#pragma unroll
      for (int sl = 0; sl < E::kShare; ++sl) {
        entry += sh_sum[sl * E::kTile + c];
        rounded += sh_max[sl * E::kTile + c];
      }
      const int64_t o = (int64_t)vt * p.part_ld + tt * E::kTile + c;
      p.part_entry[o] = entry;
      p.part_rounded[o] = rounded;
    }
  }
}

template <class E, bool kSoftcap, bool kPlain = false, bool kRounded = false>
__global__ __launch_bounds__(E::kThreads, E::kWavesPerSimd) void lce_exp_logits_panel_kernel(ExpPanelArgs p) {
  extern __shared__ __align__(16) char smem[];
  using T = typename E::T;
  static_assert(E::kHasKMajor && sizeof(T) == 2,
                "written for the four-wave direct-to-LDS engine");
  if (p.run_flag != nullptr && *p.run_flag == 0) return;
  if (p.m_dev != nullptr) {
    p.m = effective_block_rows(p.m, p.m_dev, p.row0);
    p.n_ttiles = (p.m + E::kTile - 1) / E::kTile;
  }
  int tt, vt, first_tt = 0, bid = blockIdx.x, n_ttiles = p.n_ttiles;
  if (kHasNarrowTiles<E> && p.tail_last && n_ttiles > 1 &&
      p.m - (n_ttiles - 1) * E::kTile <= 128) {
    const int before = ((n_ttiles - 1) * p.n_vtiles + kXcds - 1) / kXcds * kXcds;
    if (bid < before) {
      --n_ttiles;
    } else {
      bid -= before;
      first_tt = n_ttiles - 1;
      n_ttiles = 1;
    }
  }
  if (!xcd_tile(bid, n_ttiles, p.n_vtiles, (int64_t)E::kTile * p.h * E::kPlanes * sizeof(T), &tt,
                &vt))
    return;
  tt += first_tt;

  if constexpr (kHasNarrowTiles<E>) {
    const int tokens = p.m - tt * E::kTile;
    if (tokens <= 64) {
      exp_logits_tile<NarrowEngine<T, 2>, kSoftcap, kPlain, kRounded>(p, tt, vt, smem);
      return;
    }
    if (tokens <= 128) {
      exp_logits_tile<NarrowEngine<T, 4>, kSoftcap, kPlain, kRounded>(p, tt, vt, smem);
      return;
    }
  }
  exp_logits_tile<E, kSoftcap, kPlain, kRounded>(p, tt, vt, smem);
}

// Heads up to this size are well within the last-level cache when the narrow tiles of the last
// tokens come to read them a second time; there they come last and fill the wide tiles' last
// round.  Larger heads are read once, by neighbouring wide and narrow tiles: narrow ones alone wait
// for memory, 1.5 us a K step instead of 0.6.  Exponentiated logits in us, neighbours / last, of
// 612, 1036, 2081 and 8212 rows:
//   16 MiB  H =  256, V = 32000   36 /  33    48 /  43    73 /  69   226 / 228
//   31 MiB  H =  512, V = 32000   45 /  42    64 /  56   103 /  99   312 / 317
//   32 MiB  H = 1024, V = 16384   37 /  37    63 /  52    95 /  85   279 / 267
//   62 MiB  H = 1024, V = 32000   65 /  59    94 /  86   150 / 146   497 / 494
//   64 MiB  H = 2048, V = 16384   58 /  58   101 /  82   154 / 135   460 / 448
// Above the line it goes either way, by how the wide tiles fill whole rounds and by the cache:
//   74 MiB  H =  768, V = 50304   78 /  75   113 / 117   186 / 190   625 / 633
//   98 MiB  H = 1024, V = 50048   92 /  85   135 / 138   217 / 229   761 / 758
//  125 MiB  H = 2048, V = 32000  102 /  96   152 / 137   247 / 236
//  125 MiB  H = 1024, V = 64000   98 / 101   156 / 156   268 / 270
//  256 MiB  H = 1024, V = 131072 199 / 195   322 / 311   543 / 549   (269 rows 131 / 154)
// The line gives up gains beyond it; below, what loses loses 2 % of the kernel at most.
constexpr int64_t kTailLastWeightBytes = 64ll << 20;

template <class E, bool kSoftcap, bool kPlain = false, bool kRounded = false>
int launch_exp_panel_variant(const ExpPanelArgs& args, hipStream_t stream) {
  ExpPanelArgs a = args;
  static LdsOptIn lds;
  constexpr int kLdsBytes = kLaunchSmemBytes<E> + E::kTile * (int)sizeof(float);   // stages + stash
  if (int rc = enable_large_lds(lce_exp_logits_panel_kernel<E, kSoftcap, kPlain, kRounded>,
                                kLdsBytes, lds))
    return rc;
  a.tail_last = kHasNarrowTiles<E> && (int64_t)a.v * a.h * 2 <= kTailLastWeightBytes;
  const int grid = xcd_grid((int64_t)a.n_ttiles * a.n_vtiles) + (a.tail_last ? kXcds : 0);
  ScopedTimer timer(kClassExpPanel, stream);
  lce_exp_logits_panel_kernel<E, kSoftcap, kPlain, kRounded>
      <<<grid, E::kThreads, kLdsBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------- row kernels --
// (engine-independent; compiled beside the C ABI, reached through launch_*)

// Before the blocks: the label's logit of every row by a one-row dot product,
// which is both the loss's target term and the reference logit of the row.
struct LabelLogitArgs {
  const void* hidden;   // [m, h]
  const void* weight;   // [v, h]
  const int64_t* labels;
  int m, h, v;
  int64_t ignore, exclude;
  float softcap, logit_scale;
  float* target;        // [m] cap(scale * h . w[label]); 0 when the label has no logit
  float* ref;           // [m] reference logit; +inf for rows without loss
  float* valid_count;   // [1] rows with a label other than `ignore`
  const int64_t* m_dev = nullptr;   // device row count (null: m is exact)
  int n_count = 1;      // workgroups that count the rows (several add to a cleared valid_count)
  // what the sequence needs cleared before it, in the same launch
  int* flags = nullptr;             // [n_flags] = 0
  int n_flags = 0;
  float* losses = nullptr;          // [n_out] = 0
  int* row_of = nullptr;            // [n_out] = -1
  int64_t n_out = 0;
  // non-null (bf16): [m, h] receives the rows, zeros in place of rows without a loss (whose
  // values, NaN among them, must reach no sum over rows)
  void* rows_copy = nullptr;
  int* row_map = nullptr;           // with rows_copy: [m] the row's own index, -1 without a loss
};

struct FusedRowsArgs {
  const void* hidden;          // [m, h] rows of the block
  const int64_t* labels;       // [m]
  const float* ref;            // [m] the reference the panel was produced with
  const float* target;         // [m]
  const float* token_weights;  // [m] or null
  const int64_t* row_idx;      // [m] or null: where the row's loss goes
  int64_t loss_row0;           // row_idx == null: index of the block's first row in `losses`
  int* row_of = nullptr;       // with row_idx: row_of[row_idx[r]] = index of row r of the call
  const float* part_sum;
  const float* part_max;
  int part_ld, n_vtiles;
  int m, m_pad;                // rows of the block; rows of `scaled_hidden` to define (zeros past m)
  int h, v;
  int hp = 0;                  // float32 in planes: elements of a plane of scaled_hidden's rows
  int64_t ignore, exclude;
  float softcap, logit_scale, window;
  void* panel;                 // [.., ld], or [.., 3, ld] in planes
  int64_t ld;
  float* lse;                  // [m]
  float* losses;               // scattered, or null
  float* probabilities = nullptr;   // [m] exp(-loss), or null
  bool keep_label = false;     // the label's entry stays exp(z - c): the panel's contraction
                               // is d lse / d hidden, without the label's term
  const float* part_entry = nullptr;     // kRounded sums of the producer, or null: the row
  const float* part_rounded = nullptr;   // factor makes up for the rounding of the row's sum,
  float* row_entry = nullptr;            // [m] the sums of the row's entries, exact
  float* row_rounded = nullptr;          // [m] and rounded
  float* label_rest = nullptr;           // [m] what the label's entry lost when it was rounded
  float* row_scale;            // [m_pad]
  void* scaled_hidden;         // [m_pad, h] or [m_pad, 3, hp], or null (no grad_weight)
  float* ref_next;             // [m] reference of the second try
  int* redo;                   // [1] set when some row needs the second try
  const int* run_flag;         // non-null: run only when *run_flag != 0
  const int64_t* m_dev = nullptr;   // device row count (null: m is exact); the block's
  int64_t row0 = 0;                 // first row among the counted rows
};

// grad_hidden32[r, :] = row_scale[r] * sum over K splits of slab[s][r, :]
struct ReduceSlabsArgs {
  const float* slabs;
  int n_splits;
  int64_t split_stride;
  const float* row_scale;
  int m, h;
  float* out;   // [m, h]
  void* out_t = nullptr;            // non-null: the result goes here in bf16 instead
  const int64_t* m_dev = nullptr;   // device row count (null: m is exact); the block's
  int64_t row0 = 0;                 // first row among the counted rows
  // with a device row count the contraction derives its K splits and slab stride from
  // the real rows of the block (dynamic_k_splits); the same inputs reproduce them here
  int n_htiles = 0, tile = 0, max_splits = 1, k_steps = 0;
  int64_t slab_budget = 0;
  // non-null: row r also gets sum_j fix_value[r, j] * weight[fix_id[r, j], :] (j < kTopkFix),
  // before the row factor
  const float* fix_value = nullptr;
  const int* fix_id = nullptr;
  const float* label_rest = nullptr;     // and label_rest[r] * weight[labels[r], :]
  const int64_t* labels = nullptr;       // (read where label_rest[r] != 0)
  const void* weight = nullptr;     // bf16 [.., h]
  // non-null: one more workgroup adds up the losses (over valid_count[0] for the mean); of more
  // than kLossesPerBlock several leave their sums in loss_parts for a launch behind them
  float* loss = nullptr;
  float* loss_parts = nullptr;      // [kMaxLossParts]
  int n_parts = 1;
  int64_t part_length = 0;
  const float* losses = nullptr;    // [n_losses]
  int64_t n_losses = 0;
  const float* loss_weights = nullptr;   // non-null: sum_r loss_weights[r] * losses[loss_idx[r]]
  const int64_t* loss_idx = nullptr;     // over n_losses rows (null: r), those on the device
  const float* valid_count = nullptr;
  bool mean = false;
};
constexpr int64_t kLossesPerBlock = 16384;
constexpr int64_t kMaxLossParts = 1024;
// Largest entries of a row whose rounding the top-k path makes up for: they are known exactly
// and weigh most (a label or word of probability near 1 is most of the sum).
constexpr int kTopkFix = 8;

// out[row_idx[r], :] = dtype(g * in[r, :]) with g = grad_output[0] (/ valid_count[0]
// for the mean): the upstream gradient applied to the float32 gradients the
// forward left, rounding each entry once.
struct ScaleCastArgs {
  const float* in;          // [rows, h]
  const int64_t* row_idx;   // or null
  const float* grad_output; // [1]; reduction none: one per output row, read at row_idx[r]
  const float* valid_count; // [1], read for the mean reduction only
  int reduction;
  int64_t rows;
  int h;
  void* out;
  const int64_t* m_dev = nullptr;   // device row count: rows past it are not written
};

// scaled[r, :] = dtype(g * row_scale[r] * hidden[r, :]) with g as in ScaleCastArgs, zero
// rows from the row count up to m_pad: the K-major operand of a grad_weight
// contraction that was postponed until the upstream gradient is known.
struct ScaleRowsArgs {
  const void* hidden;       // [m, h]
  const float* row_scale;   // [m]
  const float* grad_output; // [1]; reduction none: one per output row, read at row_idx[r]
  const float* valid_count; // [1], read for the mean reduction only
  int reduction;
  int m, m_pad, h;
  void* out;                // [m_pad, h]
  const int64_t* m_dev = nullptr;   // device row count (null: m is exact)
  const int64_t* row_idx = nullptr; // output row of row r (null: r)
};

// The backward's pass over rows when the forward has left row_of: one workgroup per output
// row writes its gradient (lce_scale_cast_rows_kernel) or zeros and, when grad_weight has
// waited, the row of its operand (lce_scale_rows_kernel).
struct FinishRowsArgs {
  const float* grad_hidden32;  // [m, h]
  const int* row_of;           // [n_out] row of an output row, -1: none (null: the same row)
  bool holes = false;          // row_of is the identity but for its -1s: rows were not compacted,
                               // and the operand has zero rows in those places
  const float* grad_output;    // [1]; reduction none: [n_out]
  const float* valid_count;    // [1], read for the mean reduction only
  int reduction;
  int64_t n_out;
  int m, m_pad, h;
  const int64_t* m_dev;        // device row count (null: m is exact)
  void* grad_hidden;           // bf16 [n_out, h]
  const void* hidden = nullptr;       // [m, h], with what follows, or null
  const float* row_scale = nullptr;   // [m]
  void* scaled = nullptr;             // bf16 [m_pad, h], zero rows from the row count on
};
int launch_finish_rows(const FinishRowsArgs& a, hipStream_t stream);

// row_scale[r] = scale / sum over the vocabulary tiles of part_sum[tile][r] (0 for rows
// from m up to m_pad): the normaliser of rows whose panel holds exp(z - c).
struct SoftRowsArgs {
  const float* part_sum;
  int part_ld, n_vtiles;
  int m, m_pad;
  float scale;
  float* row_scale;
};

int launch_soft_rows(const SoftRowsArgs& a, hipStream_t stream);
// T: the operands' type, __bf16 or float (whose panel and scaled rows are in planes)
template <typename T> int launch_label_logit(LabelLogitArgs a, hipStream_t stream);
int launch_scale_rows(const ScaleRowsArgs& a, hipStream_t stream);
template <typename T> int launch_fused_rows(const FusedRowsArgs& a, hipStream_t stream);
int launch_reduce_slabs(ReduceSlabsArgs a, hipStream_t stream);
template <typename T> int launch_scale_cast(const ScaleCastArgs& a, hipStream_t stream);

// ------------------------------------------------------------------- plan ----
struct FusedPlan {
  int64_t v;
  int64_t vp;           // panel columns: the vocabulary rounded up to whole tiles
  int n_vtiles, n_htiles;
  int64_t block_rows;   // rows per block, a multiple of the tile
  int n_blocks;
  int dh_ksplit;        // K splits of the grad_hidden contraction of a full block
  int dh_max_ksplit;    // upper bound of the rule that chose them
  int64_t dh_slab_rows; // k_split_slab_rows of a full block
  int64_t k_steps;      // of its K loop, unsplit
};

// Float32 entries are three bf16 planes.
inline int panel_entry_bytes(int dtype) { return dtype == TLCE_DTYPE_F32 ? 6 : 2; }

// Cross entropies with a gradient of the head, and soft embeddings, whose panel entries are
// formed in the forward: vocabularies of whole 64-row slabs.  Others keep the sequences that
// recompute the logits, which are more exact: grad_weight contracts the hidden rows as they
// are, not a rounded product of them with a row factor, and probabilities are rounded when they
// are normalised.  2-norm errors against float64, recomputed / in the forward,
// 1500 rows, H = 1024, V = 32003: grad_weight 2.42e-3 / 2.83e-3, soft embeddings 2.25e-3 /
// 2.25e-3 (H = 3840, V = 40001, a soft cap of 30: 2.25e-3 / 2.31e-3).  A step of 2741 rows over
// H = 2048 takes 1.32 ms recomputed (1.55 from transposed copies) and took 1.04 in the forward.
// With what the label's entry and its row lose added back in float32 (1.13 ms) words that are
// labels gain, 2.1e-3 .. 2.4e-3 / 1.66e-3, and all others lose, 2.1e-3 .. 2.3e-3 / 2.5e-3 .. 2.8e-3.
inline bool fused_gradients_supported(int64_t h, int64_t v, int dtype) {
  return dtype == TLCE_DTYPE_BF16 && engine_class(h, dtype) == 2 && (v % 64) == 0;
}

// Cross entropies under a frozen head: any vocabulary.  grad_hidden is the more exact of the
// two sequences since what the label's entry loses to its rounding is added back in float32
// (lce_reduce_scaled_slabs_kernel), and two contractions replace three.  Recomputed / in the
// forward, us a step and 2-norm errors of grad_hidden against float64 (reductions mean to none):
//    600 rows, H = 1024, V = 32003    258 .. 278 / 206 .. 235   2.1e-3 .. 2.4e-3 / 1.66e-3
//   1500 rows, H = 1024, V = 32003    354 .. 382 / 260 .. 268   2.1e-3 .. 2.4e-3 / 1.66e-3
//   2741 rows, H = 2048, V = 32003   1021 .. 1036 / 727 .. 743  2.1e-3 .. 2.4e-3 / 1.66e-3
//   1610 rows, H = 4096, V = 151935        4950 / 3400
// Below 2^34 multiply-adds a contraction a step is bound by its launches (300 rows, H = 1024,
// V = 32003: 217 to 241 recomputed) and keeps its sequence.
constexpr int64_t kFrozenRaggedMinMacs = 1ll << 34;
inline bool frozen_gradients_supported(int64_t m, int64_t h, int64_t v, int dtype) {
  return fused_gradients_supported(h, v, dtype) ||
         (dtype == TLCE_DTYPE_BF16 && engine_class(h, dtype) == 2 &&
          (double)m * h * v >= (double)kFrozenRaggedMinMacs);
}

// KL and CE with top-k take any vocabulary: the contraction over it reads the rows of an
// incomplete last 64-row slab from a padded copy (k_tail_bytes).  They are the more exact
// of their two sequences (recomputed -> in the forward, same sizes: KL losses 5.4e-4 ->
// 4.5e-5, its grad_hidden 4.61e-3 -> 2.40e-3, top-k's 1.667e-3 -> 1.658e-3).
inline bool objective_gradient_in_forward_supported(int64_t h, int dtype) {
  return dtype == TLCE_DTYPE_BF16 && engine_class(h, dtype) == 2;
}

inline FusedPlan make_fused_plan(int64_t m, int64_t h, int64_t v, int dtype, int64_t panel_bytes) {
  FusedPlan p;
  p.v = v;
  const int64_t tile = 256;
  p.vp = round_up(v, tile);
  p.n_vtiles = (int)(p.vp / tile);
  p.n_htiles = (int)ceil_div(h, tile);
  if (panel_bytes <= 0) panel_bytes = kDefaultFusedPanelBytes;
  const int64_t total = ceil_div(std::max<int64_t>(m, 1), tile);   // token tiles
  const int64_t budget = std::max<int64_t>(1, panel_bytes / (p.vp * panel_entry_bytes(dtype) * tile));
  p.n_blocks = (int)ceil_div(total, budget);
  int64_t per = ceil_div(total, p.n_blocks);   // balanced blocks
  // several blocks: 16 token tiles x 16 hidden tiles make whole rounds of 256
  // workgroups in the grad_hidden contraction
  if (p.n_blocks > 1 && round_up(per, 16) <= budget) per = round_up(per, 16);
  p.block_rows = per * tile;
  p.n_blocks = (int)ceil_div(total, per);
  // (in planes, six steps of the K loop per 64 vocabulary rows)
  p.k_steps = p.vp / 64 * (dtype == TLCE_DTYPE_F32 ? SplitF32Engine::kPasses : 1);
  p.dh_max_ksplit = (int)std::max<int64_t>(1, std::min<int64_t>(kMaxKSplits, p.k_steps / 8));
  p.dh_ksplit = grad_hidden_k_splits((p.block_rows / tile) * p.n_htiles, p.dh_max_ksplit, p.k_steps,
                                     std::min(p.block_rows, std::max<int64_t>(m, 1)) * h);
  p.dh_slab_rows = k_split_slab_rows(p.dh_ksplit, p.dh_max_ksplit, (int)(p.block_rows / tile),
                                     p.n_htiles, (int)tile);
  return p;
}

// Panel budget (0: the default) of a call with a trainable head whose loss is reduced to one
// number.  In one block the panel waits for the backward, in several the float32 [v, h] sum does,
// which every block but the first reads and writes and a last pass rounds.  One block is taken
// beyond the default as well where the panel and the 16-bit gradient in the backward take no more
// than a default panel and the float32 sum in the forward, i.e. up to the default and one 16-bit
// gradient.  The step's peak then grows by no more than several blocks stay under a default panel
// (half of it at most) and by the larger block's row buffers, 6 h + v / 32 bytes for each row
// more (0.13 GB in the first line).  Several blocks / one, ms a step and GB at its peak:
//   8212 rows, H = 3840, V = 262144, cap 30   39.7 / 38.8   6.5 / 6.6
//   6000 rows, H = 4096, V = 262144           33.8 / 28.2   6.5 / 5.5    (16 and 8 token tiles)
//  10000 rows, H = 4096, V = 151936           29.8 / 27.4   5.2 / 4.7    (32 and 8)
//  16384 rows, H = 4096, V = 151936           45.0 / 43.8   5.3 / 6.6    (not taken)
inline int64_t reduced_loss_panel_bytes(int64_t m, int64_t h, int64_t v) {
  const int64_t vp = round_up(v, 256);
  const int64_t all = round_up(std::max<int64_t>(m, 1), 256) * vp * 2;
  const int64_t limit = kDefaultFusedPanelBytes + 2 * v * h;
  return all > kDefaultFusedPanelBytes && all <= limit ? all : 0;
}

struct FusedLayout {
  int64_t panel, part_sum, part_max, target, ref, ref_next, row_scale, scaled_hidden, slabs,
      redo, hidden_planes, weight_planes, label_rest, k_tail, loss_parts, total;
};

inline FusedLayout fused_layout(const FusedPlan& p, int64_t m, int64_t h, int dtype,
                                bool weight_grad) {
  FusedLayout l;
  const int64_t es = panel_entry_bytes(dtype);
  const bool planes = dtype == TLCE_DTYPE_F32;
  const int64_t hp = round_up(h, 64);   // (h itself without planes)
  const int64_t mp = round_up(std::max<int64_t>(m, 1), 256);
  int64_t off = 0;
  l.panel = off;      off += align256(p.block_rows * p.vp * es);
  l.part_sum = off;   off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.part_max = off;   off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.target = off;     off += align256(mp * 4);
  l.ref = off;        off += align256(mp * 4);
  l.ref_next = off;   off += align256(p.block_rows * 4);
  l.row_scale = off;  off += align256(p.block_rows * 4);
  l.scaled_hidden = off;
  if (weight_grad) off += align256(p.block_rows * hp * es);
  l.slabs = off;      off += align256(p.dh_slab_rows * h * 4);
  l.redo = off;       off += align256((int64_t)p.n_blocks * 4);
  l.hidden_planes = off;
  if (planes) off += align256(p.block_rows * hp * es);
  l.weight_planes = off;
  if (planes) off += align256(p.vp * hp * es);
  l.label_rest = off;
  if (!planes) off += align256(p.block_rows * 4);
  l.k_tail = off;
  if (!planes && !weight_grad) off += k_tail_bytes(p.v, h);
  l.loss_parts = off; off += align256(kMaxLossParts * 4);
  l.total = off;
  return l;
}

// The head as the K-major operand of a contraction over the vocabulary.  `k_tail`: where
// prepare_k_tail has put the rows of an incomplete last slab (null: v is a multiple of 64).
inline int prepare_k_tail(const void* weight, int64_t v, int64_t h, char* k_tail,
                          hipStream_t stream) {
  return v % 64 != 0 ? launch_k_tail(weight, v, h, k_tail, stream) : 0;
}
inline void set_head_operand(GemmArgs& g, const void* weight, int64_t v, int64_t h,
                             const char* k_tail = nullptr) {
  g.a = weight; g.lda = h; g.a_rows = (int)h;
  g.k = (int)round_up(v, 64);
  if (g.k != v) {
    g.a_tail = k_tail;
    g.a_k_full = g.k - 64;
  }
}

// Float32 cross entropies leave their gradients in the forward where they run in planes and
// the whole head's fit their bound.  Nothing is lost by it: what the row factors add are
// float32 roundings.  Per-token losses of a trainable head (whose grad_weight would have to
// wait, and the panel with it) keep the recomputing backward.  One contraction less and the
// head split once lower the sizes from which planes pay.  Forward and backward in us, float32
// engine / recomputing in planes / this (2-norm errors 2e-7 to 7e-7, on the engine 5e-7 to 3e-6):
//   1024 rows, H = 1024, V = 32000   2300 / 1439 / 1149     2048 rows  4446 / 2621 / 2017
//    512 rows, H = 2048, V = 50001   3800 / 2602 / 2071      512, H = 512, V = 16384  390 / 387 / 335
//    300 rows, H = 1024, V = 32000    992 /  -   / 668       300, H = 512, V = 16384  347 / - / 310
//    129 rows, H = 1024, V = 50001   1027 /  -   / 763       129, H = 512, V = 33000  454 / - / 388
inline bool f32_gradients_in_forward_supported(int64_t m, int64_t h, int64_t v) {
  return split_f32_supported(m, h, v, TLCE_DTYPE_F32, 128, 96) &&
         round_up(v, 256) * round_up(h, 64) * 6 <= kSplitWeightBytes;
}

// Options of the fused sequence beyond the operator's own arguments.
struct FusedOptions {
  float logit_scale = 1.0f;
  const float* token_weights = nullptr;   // [m] per-row loss weights or null
  const int64_t* row_count = nullptr;     // device int64: the real number of rows (m: capacity)
  int64_t n_out = 0;                      // entries of losses (cleared when row_idx is given)
  int* row_of = nullptr;                  // [n_out], with row_idx: LabelLogitArgs, FusedRowsArgs
  float* loss = nullptr;                  // [1]: the losses' sum, or their mean
  bool mean = false;
  void* rows_copy = nullptr;              // bf16 [m, h]: LabelLogitArgs
};

template <class E>
int fused_gradients_impl(const FusedPlan& p, const void* hidden, const void* weight,
                         const int64_t* labels, const int64_t* row_idx, int64_t m, int64_t h,
                         int64_t v, int dtype, int64_t ignore, int64_t exclude, float softcap,
                         float* losses, float* lse, float* valid_count, float* grad_hidden32,
                         float* grad_weight32, char* ws, hipStream_t stream,
                         const FusedOptions& opt) {
  // opt.row_count != null: m is the capacity every launch is sized for; the kernels
  // take the real count from the device and the workgroups past it exit at once
  const int64_t* m_dev = opt.row_count;
  using T = typename E::T;
  constexpr int kPlanes = E::kPlanes;
  using In = std::conditional_t<kPlanes == 1, T, float>;
  const bool weight_grad = grad_weight32 != nullptr;
  const FusedLayout l = fused_layout(p, m, h, dtype, weight_grad);
  T* panel = reinterpret_cast<T*>(ws + l.panel);
  float* part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  float* part_max = reinterpret_cast<float*>(ws + l.part_max);
  float* target = reinterpret_cast<float*>(ws + l.target);
  float* ref = reinterpret_cast<float*>(ws + l.ref);
  float* ref_next = reinterpret_cast<float*>(ws + l.ref_next);
  float* row_scale = reinterpret_cast<float*>(ws + l.row_scale);
  T* scaled_hidden = weight_grad ? reinterpret_cast<T*>(ws + l.scaled_hidden) : nullptr;
  float* slabs = reinterpret_cast<float*>(ws + l.slabs);
  int* redo = reinterpret_cast<int*>(ws + l.redo);
  const In* hidden_in = static_cast<const In*>(hidden);
  // the operands of the contractions, hp elements a row (and plane): the matrices
  // themselves, or their planes (of the hidden rows a block at a time)
  const int64_t hp = kPlanes == 1 ? h : round_up(h, 64);
  const T* hidden_t;
  const void* weight_t;
  if constexpr (kPlanes == 1) {
    hidden_t = hidden_in;
    weight_t = weight;
  } else {
    if (int rc = launch_split_planes(static_cast<const float*>(weight), v, p.vp, h, hp,
                                     ws + l.weight_planes, stream))
      return rc;
    hidden_t = reinterpret_cast<const T*>(ws + l.hidden_planes);
    weight_t = ws + l.weight_planes;
  }

  LabelLogitArgs la;
  la.flags = redo; la.n_flags = p.n_blocks;
  if (row_idx != nullptr) {
    la.losses = losses; la.row_of = opt.row_of; la.n_out = opt.n_out;
  }
  la.hidden = hidden; la.weight = weight; la.labels = labels;
  la.m = (int)m; la.h = (int)h; la.v = (int)v;
  la.ignore = ignore; la.exclude = exclude; la.softcap = softcap; la.logit_scale = opt.logit_scale;
  la.target = target; la.ref = ref; la.valid_count = valid_count; la.m_dev = m_dev;
  la.rows_copy = opt.rows_copy;
  la.row_map = opt.rows_copy != nullptr ? opt.row_of : nullptr;
  if (int rc = launch_label_logit<In>(la, stream)) return rc;
  if constexpr (kPlanes == 1) {
    if (opt.rows_copy != nullptr) {   // everything below reads the copy
      hidden_in = static_cast<const In*>(opt.rows_copy);
      hidden_t = hidden_in;
    }
    // (a vocabulary of incomplete slabs: frozen heads only)
    if (int rc = prepare_k_tail(weight, v, h, ws + l.k_tail, stream)) return rc;
  }
  float* label_rest = kPlanes == 1 ? reinterpret_cast<float*>(ws + l.label_rest) : nullptr;

  for (int block = 0; block < p.n_blocks; ++block) {
    const int64_t r0 = (int64_t)block * p.block_rows;
    const int64_t rows = std::min<int64_t>(p.block_rows, m - r0);
    if (rows <= 0) break;
    const int n_ttiles = (int)ceil_div(rows, E::kTile);
    const int64_t rows_p = (int64_t)n_ttiles * E::kTile;
    const int64_t rows64 = round_up(rows, 64);

    if constexpr (kPlanes > 1) {
      if (int rc = launch_split_planes(hidden_in + r0 * h, rows, rows_p, h, hp,
                                       ws + l.hidden_planes, stream))
        return rc;
    }
    ExpPanelArgs ea;
    ea.hidden = kPlanes == 1 ? hidden_t + r0 * h : hidden_t; ea.weight = weight_t;
    ea.m = (int)rows; ea.h = (int)hp; ea.v = (int)v;
    ea.exclude = exclude; ea.softcap = softcap; ea.logit_scale = opt.logit_scale;
    ea.n_ttiles = n_ttiles; ea.n_vtiles = p.n_vtiles;
    ea.panel = panel; ea.ld = p.vp;
    ea.part_sum = part_sum; ea.part_max = part_max; ea.part_ld = (int)p.block_rows;
    ea.m_dev = m_dev; ea.row0 = r0;

    FusedRowsArgs ra;
    ra.hidden = hidden_in + r0 * h; ra.labels = labels + r0;
    ra.target = target + r0;
    ra.token_weights = opt.token_weights ? opt.token_weights + r0 : nullptr;
    ra.row_idx = row_idx ? row_idx + r0 : nullptr; ra.loss_row0 = r0;
    ra.row_of = row_idx ? opt.row_of : nullptr;
    ra.part_sum = part_sum; ra.part_max = part_max;
    ra.part_ld = (int)p.block_rows; ra.n_vtiles = p.n_vtiles;
    ra.m = (int)rows; ra.m_pad = (int)rows_p; ra.h = (int)h; ra.v = (int)v; ra.hp = (int)hp;
    ra.ignore = ignore; ra.exclude = exclude; ra.softcap = softcap;
    ra.logit_scale = opt.logit_scale;
    ra.window = kRefWindow;
    ra.panel = panel; ra.ld = p.vp;
    ra.lse = lse + r0; ra.losses = losses;
    ra.row_scale = row_scale; ra.scaled_hidden = scaled_hidden;
    ra.ref_next = ref_next; ra.redo = redo + block;
    ra.m_dev = m_dev; ra.row0 = r0;
    ra.label_rest = label_rest;

    for (int attempt = 0; attempt < 2; ++attempt) {
      ea.ref = attempt ? ref_next : ref + r0;
      ea.run_flag = attempt ? redo + block : nullptr;
      if (softcap > 0.0f) {
        if (int rc = launch_exp_panel_variant<E, true>(ea, stream)) return rc;
      } else {
        if (int rc = launch_exp_panel_variant<E, false>(ea, stream)) return rc;
      }
      ra.ref = ea.ref;
      ra.run_flag = ea.run_flag;
      // the second try must not mark the block again: it reads the flag the first set
      if (int rc = launch_fused_rows<In>(ra, stream)) return rc;
    }

    // grad_hidden of the block: A = weight as stored or its planes (K-major, K = vocabulary),
    // B = panel
    GemmArgs dh;
    if constexpr (kPlanes == 1) {
      set_head_operand(dh, weight, v, h, ws + l.k_tail);
    } else {
      dh.a = weight_t; dh.lda = hp; dh.a_rows = (int)hp;
      dh.k = (int)round_up(v, 64);   // (planes have zero rows up to there)
    }
    dh.b = panel; dh.ldb = p.vp; dh.b_rows = (int)rows_p;
    dh.k_per_split = 0;
    dh.ni = p.n_htiles; dh.nj = n_ttiles;
    dh.c = slabs; dh.ldc = h; dh.c_rows = (int)rows; dh.c_cols = (int)h;
    dh.c_split_stride = p.block_rows * h;
    dh.mode = kStoreF32;
    int ksplit = (rows_p == p.block_rows)
                     ? p.dh_ksplit
                     : std::min(p.dh_ksplit,
                                grad_hidden_k_splits((int64_t)n_ttiles * p.n_htiles, p.dh_ksplit,
                                                     p.k_steps, rows * h));
    ReduceSlabsArgs rs;
    if (m_dev != nullptr) {
      // The block may hold far fewer rows than it was sized for (down to none): the kernel
      // takes as many splits as the real rows call for, within the slabs the plan allocated.
      dh.m_dev = m_dev; dh.m_role = kRowsFollow; dh.m_dev_offset = r0;
      dh.slab_budget = p.dh_slab_rows * h; dh.split_by_rows = true;
      dh.k_steps_plan = (int)p.k_steps;
      dh.max_splits = p.dh_max_ksplit;
      rs.n_htiles = p.n_htiles; rs.tile = E::kTile; rs.max_splits = dh.max_splits;
      rs.k_steps = dh.k_steps_plan; rs.slab_budget = dh.slab_budget;
    }
    if (int rc = launch_gemm<E, true, false>(dh, ksplit, kClassGradHidden, stream)) return rc;
    rs.slabs = slabs; rs.n_splits = ksplit; rs.split_stride = p.block_rows * h;
    rs.row_scale = row_scale; rs.m = (int)rows; rs.h = (int)h;
    rs.out = grad_hidden32 + r0 * h;
    rs.m_dev = m_dev; rs.row0 = r0;
    if (label_rest != nullptr) {
      rs.label_rest = label_rest; rs.labels = labels + r0; rs.weight = weight;
    }
    if (r0 + rows >= m) {
      rs.loss = opt.loss; rs.losses = losses; rs.n_losses = row_idx != nullptr ? opt.n_out : m;
      rs.valid_count = valid_count; rs.mean = opt.mean;
      rs.loss_parts = reinterpret_cast<float*>(ws + l.loss_parts);
      if (opt.loss != nullptr && opt.token_weights != nullptr) {
        rs.loss_weights = opt.token_weights; rs.loss_idx = row_idx; rs.n_losses = m;
      }
    }
    if (int rc = launch_reduce_slabs(rs, stream)) return rc;

    if (weight_grad) {
      // grad_weight += panel^T . (s * hidden): both operands K-major, K = the block's rows
      GemmArgs dw;
      dw.a = scaled_hidden; dw.lda = hp; dw.a_rows = (int)hp;
      dw.b = panel; dw.ldb = p.vp; dw.b_rows = (int)p.vp;
      dw.k = (int)rows64;
      dw.k_per_split = 0;
      dw.ni = p.n_htiles; dw.nj = p.n_vtiles;
      dw.c = grad_weight32; dw.ldc = h; dw.c_rows = (int)v; dw.c_cols = (int)h;
      dw.c_split_stride = 0;
      dw.mode = block == 0 ? kStoreF32 : kAddF32;
      dw.m_dev = m_dev; dw.m_role = kKFollows; dw.m_round = 64; dw.m_dev_offset = r0;
      if (int rc = launch_gemm<E, true, true>(dw, 1, kClassGradWeight, stream)) return rc;
    }
  }
  return 0;
}

// The grad_weight contraction of a single-block forward, postponed to the backward:
// when all rows fit one block the panel still holds every exp(z - c) after the forward,
// so grad_weight = panel^T . (g * s * hidden) can be formed once the upstream gradient
// g is known and stored directly in the input dtype: no float32 [v, h] accumulator
// and no pass that scales and rounds it.  `ws` is the forward's workspace, untouched
// since (the forward was called without a grad_weight buffer, as for a frozen head,
// on a workspace sized for one).
template <class E>
int deferred_contraction(const FusedPlan& p, const FusedLayout& l, int64_t m, int64_t h, int64_t v,
                         const int64_t* m_dev, void* grad_weight, char* ws, hipStream_t stream) {
  using T = typename E::T;
  GemmArgs dw;
  dw.a = ws + l.scaled_hidden; dw.lda = h; dw.a_rows = (int)h;
  dw.b = ws + l.panel; dw.ldb = p.vp; dw.b_rows = (int)p.vp;
  dw.k = (int)round_up(m, 64);
  dw.k_per_split = 0;
  dw.ni = p.n_htiles; dw.nj = p.n_vtiles;
  dw.c = static_cast<T*>(grad_weight); dw.ldc = h; dw.c_rows = (int)v; dw.c_cols = (int)h;
  dw.c_split_stride = 0;
  dw.mode = kStoreT;
  dw.m_dev = m_dev; dw.m_role = kKFollows; dw.m_round = 64;
  return launch_gemm<E, true, true>(dw, 1, kClassGradWeight, stream);
}

template <class E>
int deferred_grad_weight_impl(const FusedPlan& p, const void* hidden, int64_t m, int64_t h,
                              int64_t v, int dtype, const float* grad_output,
                              const float* valid_count, int reduction, const int64_t* m_dev,
                              const int64_t* row_idx, void* grad_weight, char* ws,
                              hipStream_t stream) {
  const FusedLayout l = fused_layout(p, m, h, dtype, true);
  const int64_t rows_p = round_up(m, E::kTile);
  ScaleRowsArgs sa;
  sa.hidden = hidden; sa.row_scale = reinterpret_cast<const float*>(ws + l.row_scale);
  sa.grad_output = grad_output; sa.valid_count = valid_count; sa.reduction = reduction;
  sa.m = (int)m; sa.m_pad = (int)rows_p; sa.h = (int)h;
  sa.out = ws + l.scaled_hidden; sa.m_dev = m_dev; sa.row_idx = row_idx;
  if (int rc = launch_scale_rows(sa, stream)) return rc;
  return deferred_contraction<E>(p, l, m, h, v, m_dev, grad_weight, ws, stream);
}

// Soft embedding under a soft cap in two contractions instead of three
// (streaming_soft_embedding.py:60-148 computes softmax(cap(h W^T)) W with running
// maxima over vocabulary chunks): capped logits lie in [-cap, cap], so exp(z - cap)
// lies in [exp(-2 cap), 1] and needs no row maximum.  Per block of rows over the whole
// vocabulary: the panel receives exp(z - cap) in bf16 and the per-tile sums go out as
// partials, then out[r, :] = (scale / sum_r) * (panel . weight)[r, :] in float32,
// rounded once.  cap <= kSoftEmbeddingMaxCap keeps exp(-2 cap) a normal bf16 number.
constexpr float kSoftEmbeddingMaxCap = 40.0f;

template <class E>
int soft_embedding_fused_impl(const FusedPlan& p, const void* hidden, const void* weight,
                              int64_t m, int64_t h, int64_t v, int dtype, float softcap,
                              float scale, void* out, char* ws, hipStream_t stream) {
  using T = typename E::T;
  const FusedLayout l = fused_layout(p, m, h, dtype, false);
  T* panel = reinterpret_cast<T*>(ws + l.panel);
  float* part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  float* part_max = reinterpret_cast<float*>(ws + l.part_max);
  float* row_scale = reinterpret_cast<float*>(ws + l.row_scale);
  float* slabs = reinterpret_cast<float*>(ws + l.slabs);
  const T* hidden_t = static_cast<const T*>(hidden);
  for (int block = 0; block < p.n_blocks; ++block) {
    const int64_t r0 = (int64_t)block * p.block_rows;
    const int64_t rows = std::min<int64_t>(p.block_rows, m - r0);
    if (rows <= 0) break;
    const int n_ttiles = (int)ceil_div(rows, E::kTile);
    const int64_t rows_p = (int64_t)n_ttiles * E::kTile;

    ExpPanelArgs ea;
    ea.hidden = hidden_t + r0 * h; ea.weight = weight;
    ea.ref = nullptr; ea.ref_const = softcap;
    ea.m = (int)rows; ea.h = (int)h; ea.v = (int)v;
    ea.exclude = -1; ea.softcap = softcap; ea.logit_scale = 1.0f;
    ea.n_ttiles = n_ttiles; ea.n_vtiles = p.n_vtiles;
    ea.panel = panel; ea.ld = p.vp;
    ea.part_sum = part_sum; ea.part_max = part_max; ea.part_ld = (int)p.block_rows;
    ea.run_flag = nullptr;
    if (int rc = launch_exp_panel_variant<E, true, true>(ea, stream)) return rc;

    SoftRowsArgs sr;
    sr.part_sum = part_sum; sr.part_ld = (int)p.block_rows; sr.n_vtiles = p.n_vtiles;
    sr.m = (int)rows; sr.m_pad = (int)rows_p; sr.scale = scale; sr.row_scale = row_scale;
    if (int rc = launch_soft_rows(sr, stream)) return rc;

    // the contraction of grad_hidden in the forward that leaves the gradients: K = the
    // vocabulary, K splits into slabs for few rows
    GemmArgs g;
    set_head_operand(g, weight, v, h);
    g.b = panel; g.ldb = p.vp; g.b_rows = (int)rows_p;
    g.k_per_split = 0;
    g.ni = p.n_htiles; g.nj = n_ttiles;
    g.c = slabs; g.ldc = h; g.c_rows = (int)rows; g.c_cols = (int)h;
    g.c_split_stride = p.block_rows * h;
    g.mode = kStoreF32;
    const int ksplit = (rows_p == p.block_rows)
                           ? p.dh_ksplit
                           : std::min(p.dh_ksplit,
                                      grad_hidden_k_splits((int64_t)n_ttiles * p.n_htiles,
                                                           p.dh_ksplit, p.vp / 64, rows * h));
    if (int rc = launch_gemm<E, true, false>(g, ksplit, kClassGradHidden, stream)) return rc;
    ReduceSlabsArgs rs;
    rs.slabs = slabs; rs.n_splits = ksplit; rs.split_stride = p.block_rows * h;
    rs.row_scale = row_scale; rs.m = (int)rows; rs.h = (int)h;
    rs.out = nullptr; rs.out_t = static_cast<T*>(out) + r0 * h;
    if (int rc = launch_reduce_slabs(rs, stream)) return rc;
  }
  return 0;
}

// ---- frozen-head cross entropy with top-k: the gradient formed in the forward ----
// Two ways.  Through exponentiated logits (topk_from_exp_impl): the pass over the head is
// the cross entropy's, entries exp(z - label's logit)*cap' in bf16 and exact float32 maxima of
// every 256-word tile; no float32 logits cross memory.  lce_topk_select_kernel finds the k
// largest logits from them: the k-th largest tile maximum bounds the k-th largest logit from
// below, so only tiles that reach it are read (about k of them), entries above the bound are
// candidates, and the logits of the few that remain are computed again in float32, one dot
// product each.  Rows that this cannot settle (more near-ties than it has room for, top
// logits so far below the label's that their entries underflow) raise a flag, on which the
// second way's panels and scan run for the block, lists only.
//
// What the rows lose by a reference other than their maximum (whose entry would be 1 exactly)
// they get back twice: the kTopkFix largest entries' errors, which are known once their logits
// are, are added to the contraction's row, and the row factor takes out the part of the
// rounding errors that the other entries share.
// d lse / d hidden against float64, the other way -> this (1100 rows, H = 512, V = 32000, label
// logits raised by 0 / 8 / 12): 4.89e-4, 9.95e-5, 3.29e-6 -> 4.88e-4, 9.90e-5, 3.46e-6 (a factor for
// all entries 4.01e-6 there); with a soft cap of 30 (2100 rows, H = 1024, V = 50001) 4.39e-4,
// 9.88e-4, 1.32e-3 -> 4.37e-4, 1.61e-4, 8.9e-6; head rows with a common mean 1.43e-5 -> 9.8e-6.
//
// Measured on 8192 rows, H = 4096, V = 151936, k = 16, forward and backward: 18.5 -> 15.2 ms: the
// pass over the head 8.1 -> 7.6, the scan's 2.1, the entries' 1.4 and their rescaling's 0.4 ->
// 0.25 for the selection and 0.1 for the corrections.
//
// Through float32 logits (the rest of this comment), for few tiles per top-k entry:
// The backward of tlce_ce_topk_* recomputes the logits to form the softmax panel
// (3 contractions per step).  Here the forward, which stages float32 logits panels
// anyway, also writes e = exp(z - reference) * cap' of every panel in bf16 into a
// panel over the whole vocabulary and contracts it with the weight rows once:
//   unit[r, :] = (multiplier / sum_r) * (e . weight)[r, :] = d lse_r / d hidden[r, :]
// (2 contractions).  The reference of a panel is the row's largest logit so far (known
// after the panel's scan), so e <= 1; panels written before a row's maximum grew are
// multiplied by exp(old - final) afterwards (lce_rescale_exp_rows_kernel).  The
// backward is then one pass over rows: ce_scale[r] * unit[r, :] plus the single-row
// terms of the label and the top-k ids, rounded once.
struct RescaleExpArgs {
  void* panel;             // bf16 [m_pad, ld]
  int64_t ld;
  int m, m_pad;
  const float* ref_used;   // [n_panels, m_pad]
  const float* run_max;    // [m] the final row maxima
  int64_t panel_width;     // columns per logits panel
  int64_t total_width;     // columns of the whole panel
};

struct TopkRowScaleArgs {
  const float* run_sum;    // [m] sum of exp(z - max)
  float multiplier;
  int m, m_pad;
  float* row_scale;        // [m_pad] multiplier / sum; 0 from m on
};

struct TopkApplyArgs {
  const float* unit;       // [m, h] d lse / d hidden
  const void* hidden;
  const void* weight;
  const int64_t* labels;
  const int64_t* top_ids;          // [m, k]; outside [0, v): no word (TopkAdjustArgs)
  const float* ce_scale;           // [m]
  const float* grad_top_values;    // [m, k] or null
  int m, h, v, k;
  float softcap, logit_scale;
  void* grad_hidden;               // bf16 [m, h]
};

int launch_rescale_exp_rows(const RescaleExpArgs& a, int n_panels, hipStream_t stream);
int launch_topk_row_scale(const TopkRowScaleArgs& a, hipStream_t stream);
int launch_topk_apply(const TopkApplyArgs& a, hipStream_t stream);

struct TopkSelectArgs {
  const void* panel;       // bf16 [.., ld] exp(z - ref) * cap'
  int64_t ld;
  const float* part_max;   // [n_vtiles, part_ld] base-2 tile maxima of z
  int part_ld, n_vtiles;
  const float* ref;        // [m] the label's logit; ref_next where *redo
  const float* ref_next;
  const int* redo;
  const void* hidden;      // [m, h]
  const void* weight;      // [v, h]
  int m, h, k;
  float softcap, logit_scale;
  float* top_values;       // [m, k]
  int64_t* top_ids;        // [m, k]
  int* unsettled;          // set when some row's list could not be found
  // the largest entries (kTopkFix, at most k): what takes their exact values' place, and the
  // row factor that makes up for the rounding of the other entries' sum
  float* fix_value;        // [m, kTopkFix]
  int* fix_id;             // [m, kTopkFix]
  const float* row_entry;     // [m] sum of the row's entries
  const float* row_rounded;   // [m] sum of the row's rounded entries
  float* row_scale;        // [m]
};
int launch_topk_select(const TopkSelectArgs& a, hipStream_t stream);

// Tiles whose maxima a wave holds; the k-th largest of them is a useful bound while there
// are some per list entry.
constexpr int kTopkSelectTiles = 1024;
// Below 2^25 logits the step is bound by the host's launches, of which there are more here
// (ms, float32 logits / this: 300 rows, V = 16384 0.335 / 0.345; 1024, V = 20000 0.335 / 0.350;
// 1024 rows, H = 2048, V = 33000 0.593 / 0.524; 4096, H = 1024, V = 32768, k = 64 1.38 / 0.92).
inline bool topk_from_exp_supported(int64_t m, int64_t v, int top_k) {
  const int64_t tiles = ceil_div(v, 256);
  if (m * v < (1ll << 25)) return false;
  return tiles <= kTopkSelectTiles && tiles >= std::max<int64_t>(64, 2 * top_k);
}

struct TopkFusedLayout {
  int64_t forward, panel, ref_used, row_scale, slabs, k_tail, part_sum, part_max, part_entry,
      part_rounded, target, ref, ref_next, row_entry, row_rounded, fix_value, fix_id, flags, total;
};

// Rows are taken in blocks of the panel budget of the forward that leaves the gradients
// (its default; panel_bytes bounds the float32 logits panels here): rows are independent,
// so a block is a call of its own on a part of every per-row buffer.
inline bool topk_gradient_in_forward_supported(int64_t m, int64_t h, int64_t v, int dtype) {
  (void)m;
  (void)v;
  return objective_gradient_in_forward_supported(h, dtype);
}

// Rows per block of the objectives that take whole blocks of rows one after the other.
inline int64_t fused_row_block(int64_t m, int64_t h, int64_t v, int dtype) {
  return make_fused_plan(m, h, v, dtype, 0).block_rows;
}

inline TopkFusedLayout topk_fused_layout(const TopkPlan& t, const FusedPlan& p, int64_t h) {
  TopkFusedLayout l;
  int64_t off = 0;
  l.forward = off;    off += align256(t.forward_total);
  l.panel = off;      off += align256(p.block_rows * p.vp * 2);
  l.ref_used = off;   off += align256((int64_t)t.n_fpanels * p.block_rows * 4);
  l.row_scale = off;  off += align256(p.block_rows * 4);
  l.slabs = off;      off += align256((int64_t)p.dh_ksplit * p.block_rows * h * 4);
  l.k_tail = off;     off += k_tail_bytes(p.v, h);
  l.part_sum = off;   off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.part_max = off;   off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.part_entry = off; off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.part_rounded = off; off += align256((int64_t)p.n_vtiles * p.block_rows * 4);
  l.target = off;     off += align256(p.block_rows * 4);
  l.ref = off;        off += align256(p.block_rows * 4);
  l.ref_next = off;   off += align256(p.block_rows * 4);
  l.row_entry = off;  off += align256(p.block_rows * 4);
  l.row_rounded = off; off += align256(p.block_rows * 4);
  l.fix_value = off;  off += align256(p.block_rows * kTopkFix * 4);
  l.fix_id = off;     off += align256(p.block_rows * kTopkFix * 4);
  l.flags = off;      off += 256;   // redo, unsettled, count of rows (unused)
  l.total = off;
  return l;
}

// unit[r, :] = row_scale[r] * (panel . weight)[r, :]
template <class E>
int topk_contraction(const TopkFusedLayout& l, const FusedPlan& p, const void* weight, int64_t m,
                     int64_t h, int64_t v, float* unit_grad, char* ws, hipStream_t stream,
                     bool fix = false) {
  const int m_pad = (int)p.block_rows;
  float* slabs = reinterpret_cast<float*>(ws + l.slabs);
  if (int rc = prepare_k_tail(weight, v, h, ws + l.k_tail, stream)) return rc;
  GemmArgs g;
  set_head_operand(g, weight, v, h, ws + l.k_tail);
  g.b = ws + l.panel; g.ldb = p.vp; g.b_rows = m_pad;
  g.k_per_split = 0;
  g.ni = p.n_htiles; g.nj = m_pad / E::kTile;
  g.c = slabs; g.ldc = h; g.c_rows = (int)m; g.c_cols = (int)h;
  g.c_split_stride = p.block_rows * h;
  g.mode = kStoreF32;
  if (int rc = launch_gemm<E, true, false>(g, p.dh_ksplit, kClassGradHidden, stream)) return rc;
  ReduceSlabsArgs rs;
  rs.slabs = slabs; rs.n_splits = p.dh_ksplit; rs.split_stride = p.block_rows * h;
  rs.row_scale = reinterpret_cast<const float*>(ws + l.row_scale);
  rs.m = (int)m; rs.h = (int)h;
  rs.out = unit_grad;
  if (fix) {
    rs.fix_value = reinterpret_cast<const float*>(ws + l.fix_value);
    rs.fix_id = reinterpret_cast<const int*>(ws + l.fix_id);
    rs.weight = weight;
  }
  return launch_reduce_slabs(rs, stream);
}

template <class E>
int topk_from_exp_impl(const TopkPlan& t, const FusedPlan& p, const void* hidden,
                       const void* weight, const int64_t* labels, int64_t m, int64_t h, int64_t v,
                       int top_k, float multiplier, float softcap, float* losses,
                       float* probabilities, float* top_values, int64_t* top_ids, float* lse,
                       float* unit_grad, char* ws, hipStream_t stream) {
  const TopkFusedLayout l = topk_fused_layout(t, p, h);
  constexpr int64_t kNoIgnore = INT64_MIN;   // every row has a loss
  float* target = reinterpret_cast<float*>(ws + l.target);
  float* ref = reinterpret_cast<float*>(ws + l.ref);
  float* ref_next = reinterpret_cast<float*>(ws + l.ref_next);
  int* redo = reinterpret_cast<int*>(ws + l.flags);
  int* unsettled = redo + 1;
  LabelLogitArgs la;
  la.flags = redo; la.n_flags = 2;
  la.hidden = hidden; la.weight = weight; la.labels = labels;
  la.m = (int)m; la.h = (int)h; la.v = (int)v;
  la.ignore = kNoIgnore; la.exclude = -1; la.softcap = softcap; la.logit_scale = multiplier;
  la.target = target; la.ref = ref; la.valid_count = reinterpret_cast<float*>(redo + 2);
  if (int rc = launch_label_logit<typename E::T>(la, stream)) return rc;

  ExpPanelArgs ea;
  ea.hidden = hidden; ea.weight = weight;
  ea.m = (int)m; ea.h = (int)h; ea.v = (int)v;
  ea.exclude = -1; ea.softcap = softcap; ea.logit_scale = multiplier;
  ea.n_ttiles = (int)(p.block_rows / E::kTile); ea.n_vtiles = p.n_vtiles;
  ea.panel = ws + l.panel; ea.ld = p.vp;
  ea.part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  ea.part_max = reinterpret_cast<float*>(ws + l.part_max);
  ea.part_ld = (int)p.block_rows;
  ea.part_entry = reinterpret_cast<float*>(ws + l.part_entry);
  ea.part_rounded = reinterpret_cast<float*>(ws + l.part_rounded);
  FusedRowsArgs ra;
  ra.part_entry = ea.part_entry; ra.part_rounded = ea.part_rounded;
  ra.row_entry = reinterpret_cast<float*>(ws + l.row_entry);
  ra.row_rounded = reinterpret_cast<float*>(ws + l.row_rounded);
  ra.hidden = hidden; ra.labels = labels; ra.target = target; ra.token_weights = nullptr;
  ra.row_idx = nullptr; ra.loss_row0 = 0;
  ra.part_sum = ea.part_sum; ra.part_max = ea.part_max;
  ra.part_ld = ea.part_ld; ra.n_vtiles = p.n_vtiles;
  ra.m = (int)m; ra.m_pad = (int)p.block_rows; ra.h = (int)h; ra.v = (int)v;
  ra.ignore = kNoIgnore; ra.exclude = -1; ra.softcap = softcap; ra.logit_scale = multiplier;
  ra.window = kRefWindow;
  ra.panel = ea.panel; ra.ld = ea.ld;
  ra.lse = lse; ra.losses = losses; ra.probabilities = probabilities; ra.keep_label = true;
  ra.row_scale = reinterpret_cast<float*>(ws + l.row_scale); ra.scaled_hidden = nullptr;
  ra.ref_next = ref_next; ra.redo = redo;
  for (int attempt = 0; attempt < 2; ++attempt) {
    ea.ref = ra.ref = attempt ? ref_next : ref;
    ea.run_flag = ra.run_flag = attempt ? redo : nullptr;
    if (softcap > 0.0f) {
      if (int rc = launch_exp_panel_variant<E, true, false, true>(ea, stream)) return rc;
    } else {
      if (int rc = launch_exp_panel_variant<E, false, false, true>(ea, stream)) return rc;
    }
    if (int rc = launch_fused_rows<typename E::T>(ra, stream)) return rc;
  }

  TopkSelectArgs sa;
  sa.panel = ea.panel; sa.ld = ea.ld;
  sa.part_max = ea.part_max; sa.part_ld = ea.part_ld; sa.n_vtiles = p.n_vtiles;
  sa.ref = ref; sa.ref_next = ref_next; sa.redo = redo;
  sa.hidden = hidden; sa.weight = weight;
  sa.m = (int)m; sa.h = (int)h; sa.k = top_k; sa.softcap = softcap; sa.logit_scale = multiplier;
  sa.top_values = top_values; sa.top_ids = top_ids; sa.unsettled = unsettled;
  sa.fix_value = reinterpret_cast<float*>(ws + l.fix_value);
  sa.fix_id = reinterpret_cast<int*>(ws + l.fix_id);
  sa.row_entry = ra.row_entry; sa.row_rounded = ra.row_rounded; sa.row_scale = ra.row_scale;
  if (int rc = launch_topk_select(sa, stream)) return rc;
  if (int rc = topk_forward_impl<E>(t, hidden, weight, labels, m, h, v, top_k, multiplier, softcap,
                                    losses, probabilities, top_values, top_ids, lse,
                                    ws + l.forward, stream, nullptr, unsettled))
    return rc;
  return topk_contraction<E>(l, p, weight, m, h, v, unit_grad, ws, stream, true);
}

template <class E>
int topk_forward_with_gradient_impl(const TopkPlan& t, const FusedPlan& p, const void* hidden,
                                    const void* weight, const int64_t* labels, int64_t m,
                                    int64_t h, int64_t v, int top_k, float multiplier,
                                    float softcap, float* losses, float* probabilities,
                                    float* top_values, int64_t* top_ids, float* lse,
                                    float* unit_grad, char* ws, hipStream_t stream) {
  using T = typename E::T;
  if (topk_from_exp_supported(m, v, top_k))
    return topk_from_exp_impl<E>(t, p, hidden, weight, labels, m, h, v, top_k, multiplier, softcap,
                                 losses, probabilities, top_values, top_ids, lse, unit_grad, ws,
                                 stream);
  const TopkFusedLayout l = topk_fused_layout(t, p, h);
  char* fws = ws + l.forward;
  T* panel = reinterpret_cast<T*>(ws + l.panel);
  float* ref_used = reinterpret_cast<float*>(ws + l.ref_used);
  float* row_scale = reinterpret_cast<float*>(ws + l.row_scale);
  const int m_pad = (int)p.block_rows;
  TopkExpHook hook;
  hook.panel = panel; hook.ld = p.vp; hook.m_pad = m_pad; hook.ref_used = ref_used;
  if (int rc = topk_forward_impl<E>(t, hidden, weight, labels, m, h, v, top_k, multiplier,
                                    softcap, losses, probabilities, top_values, top_ids, lse,
                                    fws, stream, &hook))
    return rc;
  const float* run_max = reinterpret_cast<const float*>(fws + t.run_max);
  const float* run_sum = reinterpret_cast<const float*>(fws + t.run_sum);
  if (t.n_fpanels > 1) {
    RescaleExpArgs ra;
    ra.panel = panel; ra.ld = p.vp; ra.m = (int)m; ra.m_pad = m_pad;
    ra.ref_used = ref_used; ra.run_max = run_max;
    ra.panel_width = t.vcf; ra.total_width = p.vp;
    if (int rc = launch_rescale_exp_rows(ra, t.n_fpanels - 1, stream)) return rc;
  }
  TopkRowScaleArgs sa;
  sa.run_sum = run_sum; sa.multiplier = multiplier; sa.m = (int)m; sa.m_pad = m_pad;
  sa.row_scale = row_scale;
  if (int rc = launch_topk_row_scale(sa, stream)) return rc;
  return topk_contraction<E>(l, p, weight, m, h, v, unit_grad, ws, stream);
}

// ---- frozen-head KL: the gradient formed in the forward (3 contractions, not 6) ----
// A pass over a head holds every logit of a tile in registers.  The emitting variant of
// the KL panel kernel (lce_kl_panel_kernel<.., kEmit>) finds the exact maximum of each
// token over the tile's 256 vocabulary rows and writes e = exp2(z2 - tile maximum) <= 1
// in bf16 into a panel over the whole vocabulary, beside the tile's softmax partials:
// softmax = e * exp2(tile maximum - lse2) per (token, tile) once the lse is known, and
// nothing has to be known beforehand.  One such pass over the teacher head (no teacher
// tile to read: kNoTeacher) replaces its statistics pass and its probabilities pass;
// the draft pass reads the teacher's entries, scales them to probabilities per (token,
// tile), accumulates the loss terms and emits its own entries.  One elementwise pass
// then turns the two panels into the logit gradient
//   g[r, v] = e_d * exp2(max_d[tile, r] - lse2_d[r]) - e_t * exp2(max_t[tile, r] - lse2_t[r])
// (lce_kl_grad_from_exp_kernel), and one contraction with the draft head leaves
//   unit[r, :] = d loss[r] / d draft_hidden[r, :]       float32 [m, h].
// The backward multiplies row r by its upstream gradient and rounds once.  Under a soft
// cap the gradient also carries cap'(z) = 1 - (z / cap)^2, with z re-derived from the
// entry (z2 = log2(entry) + tile maximum; the rounding of the entry moves z by less than
// 0.003); a cap of at most kSoftEmbeddingMaxCap keeps every entry a normal bf16 number.
struct KlGradFromExpArgs {
  void* exp_panel;           // bf16 [mp, ld]: e in, logit gradient out
  const void* teacher;       // bf16 [mp, ld] teacher probabilities
  int64_t ld;
  int m, mp;
  const float* part_max;     // [n_vtiles, part_ld] base-2 tile maxima of the draft
  int part_ld;
  const float* draft_lse;    // [m] natural units
  float softcap = 0.0f;      // > 0: the gradient is multiplied by cap'(z)
  const float* t_part_max = nullptr;   // non-null: `teacher` holds entries of the same kind,
  const float* t_lse = nullptr;        // these are the teacher's tile maxima and lse
  // teacher == null: the entries are only normalised (softmax of the rows, times
  // exp(-draft_lse offset) if the caller folded a factor into draft_lse)
};

// lse[r] - log(scale) from the per-tile (maximum, sum) partials of an emitting pass
// (so that exp2(tile maximum - lse2) carries the factor `scale`), and row_scale = 1
// (0 from m on) for the slab reduction that follows.
struct EmitRowsArgs {
  const float* part_max;   // [n_vtiles, part_ld] base-2 tile maxima
  const float* part_sum;   // [n_vtiles, part_ld] sums of exp2(z2 - tile maximum)
  int part_ld, n_vtiles;
  int m, m_pad;
  float scale;             // > 0
  float* lse;              // [m_pad]
  float* row_scale;        // [m_pad]
};
int launch_emit_rows(const EmitRowsArgs& a, hipStream_t stream);
int launch_kl_grad_from_exp(const KlGradFromExpArgs& a, int n_vtiles, hipStream_t stream);

constexpr float kKlMinCap = 10.0f;

struct KlFusedLayout {
  int64_t kl, teacher_parts, teacher, exp_panel, slabs, k_tail, total;
};

template <class E, bool kSoftcap, bool kNoTeacher>
int launch_kl_panel_emit_variant(const KlPanelArgs& a, hipStream_t stream) {
  static LdsOptIn lds;
  constexpr int kLdsBytes = E::kSmemBytes + E::kShare * E::kTile * (int)sizeof(float);
  if (int rc = enable_large_lds(lce_kl_panel_kernel<E, kSoftcap, false, true, kNoTeacher>,
                                kLdsBytes, lds))
    return rc;
  const int grid = xcd_grid((int64_t)a.n_ttiles * a.n_ptiles);
  ScopedTimer timer(kClassGradLogits, stream);
  lce_kl_panel_kernel<E, kSoftcap, false, true, kNoTeacher>
      <<<grid, E::kThreads, kLdsBytes, stream>>>(a);
  TLCE_LAUNCH_CHECK();
  return 0;
}

// panel_in == null: the pass over a head on its own (no teacher tile is read)
template <class E>
int launch_kl_panel_emit(const KlPanelArgs& a, hipStream_t stream) {
  if (a.panel_in == nullptr) {
    return a.softcap > 0.0f ? launch_kl_panel_emit_variant<E, true, true>(a, stream)
                            : launch_kl_panel_emit_variant<E, false, true>(a, stream);
  }
  return a.softcap > 0.0f ? launch_kl_panel_emit_variant<E, true, false>(a, stream)
                          : launch_kl_panel_emit_variant<E, false, false>(a, stream);
}

inline bool kl_gradient_in_forward_supported(int64_t m, int64_t hd, int64_t ht, int64_t v,
                                             int dtype, float softcap) {
  (void)m;   // rows beyond one block of the panel budget are taken block by block
  // cap'(z) is re-derived from entries rounded to bf16, which moves z by up to 0.003 and
  // cap' = 1 - (z / cap)^2 by up to 0.006 / cap: negligible beside the entries whose cap'
  // is of order one, but under a small cap with every logit deep in it nothing else is
  // left (measured: 2 % of the gradient's largest entry at cap 3): caps below 10 keep the
  // sequence that evaluates cap' on the float32 logit
  const bool cap_ok = softcap <= 0.0f || (softcap >= kKlMinCap && softcap <= kSoftEmbeddingMaxCap);
  (void)v;
  return cap_ok && objective_gradient_in_forward_supported(hd, dtype) && engine_class(ht, dtype) == 2;
}

inline KlFusedLayout kl_fused_layout(const KlLayout& kl, const Plan& pd, const FusedPlan& p,
                                     int64_t hd) {
  KlFusedLayout l;
  int64_t off = 0;
  l.kl = off;         off += align256(kl.total);
  l.teacher_parts = off;  off += 2 * kl.tile_part;
  l.teacher = off;    off += align256(pd.mp * pd.vp * 2);
  l.exp_panel = off;  off += align256(pd.mp * pd.vp * 2);
  l.slabs = off;      off += align256((int64_t)p.dh_ksplit * pd.mp * hd * 4);
  l.k_tail = off;     off += k_tail_bytes(p.v, hd);
  l.total = off;
  return l;
}

template <class E>
int kl_forward_with_gradient_impl(const Plan& pd, const Plan& pt, const KlLayout& kl,
                                  const FusedPlan& fp, const void* draft_hidden,
                                  const void* draft_weight, const void* teacher_hidden,
                                  const void* teacher_weight, int64_t m, int64_t hd, int64_t ht,
                                  int64_t v, int dtype, float softcap, float* losses,
                                  float* draft_lse, float* teacher_lse, float* unit_grad,
                                  char* ws, hipStream_t stream) {
  using T = typename E::T;
  const KlFusedLayout l = kl_fused_layout(kl, pd, fp, hd);
  char* kws = ws + l.kl;
  T* teacher = reinterpret_cast<T*>(ws + l.teacher);
  T* exp_panel = reinterpret_cast<T*>(ws + l.exp_panel);
  float* slabs = reinterpret_cast<float*>(ws + l.slabs);
  float* part_max = reinterpret_cast<float*>(kws + kl.stats);
  float* part_sum = reinterpret_cast<float*>(kws + kl.stats + kl.tile_part);
  float* loss_part = reinterpret_cast<float*>(kws + kl.stats + 2 * kl.tile_part);
  float* tsum_part = reinterpret_cast<float*>(kws + kl.stats + 3 * kl.tile_part);
  float* t_part_max = reinterpret_cast<float*>(ws + l.teacher_parts);
  float* t_part_sum = reinterpret_cast<float*>(ws + l.teacher_parts + kl.tile_part);
  float* ones = reinterpret_cast<float*>(kws + kl.ones);
  (void)pt;
  ScaleArgs sa;
  sa.labels = nullptr; sa.row_idx = nullptr; sa.grad_output = nullptr; sa.valid_count = nullptr;
  sa.m = (int)m; sa.mp = (int)pd.mp; sa.reduction = TLCE_REDUCTION_SUM; sa.ignore = 0;
  sa.scale = ones; sa.constant = 1.0f; sa.multiplier = 1.0f;
  if (int rc = launch_token_scale(sa, stream)) return rc;

  auto lse_from_partials = [&](const void* hidden, const void* weight, int64_t h,
                               const float* pmax, const float* psum, float* lse) -> int {
    CombineArgs ca;
    ca.hidden = hidden; ca.weight = weight; ca.bias = nullptr; ca.labels = nullptr;
    ca.row_idx = nullptr;
    ca.m = (int)m; ca.h = (int)h; ca.v = (int)v;
    ca.ignore = 0; ca.exclude = -1; ca.softcap = softcap;
    ca.part_max = pmax; ca.part_sum = psum;
    ca.part_ld = (int)pd.mp; ca.nsplit = pd.n_vtiles;
    ca.losses = nullptr; ca.lse = lse; ca.valid_count = nullptr;
    ca.label_offset = 0; ca.local_max = nullptr; ca.local_sum = nullptr;
    ca.target_logits = nullptr;
    ScopedTimer timer(kClassCombine, stream);
    lce_combine_loss_kernel<T><<<(int)ceil_div(m, kCombineRowsPerBlock),
                                64 * kCombineRowsPerBlock, 0, stream>>>(ca);
    TLCE_LAUNCH_CHECK();
    return 0;
  };

  KlPanelArgs ka;
  ka.lse = nullptr; ka.scale = nullptr;
  ka.m = (int)m; ka.v = (int)v; ka.softcap = softcap;
  ka.v0 = 0; ka.n_ttiles = pd.n_ttiles; ka.n_ptiles = pd.n_vtiles;
  ka.ld = pd.vp; ka.part_ld = (int)pd.mp; ka.mode = kKlLoss;
  ka.loss_part = loss_part; ka.tsum_part = tsum_part;
  // the teacher head on its own: entries and softmax partials in one contraction
  ka.hidden = teacher_hidden; ka.weight = teacher_weight; ka.h = (int)ht;
  ka.panel = teacher; ka.panel_in = nullptr;
  ka.part_max = t_part_max; ka.part_sum = t_part_sum;
  if (int rc = launch_kl_panel_emit<E>(ka, stream)) return rc;
  if (int rc = lse_from_partials(teacher_hidden, teacher_weight, ht, t_part_max, t_part_sum,
                                 teacher_lse))
    return rc;
  // the draft head against it: loss terms, softmax partials and its own entries
  ka.hidden = draft_hidden; ka.weight = draft_weight; ka.h = (int)hd;
  ka.panel = exp_panel; ka.panel_in = teacher; ka.ld_in = pd.vp;
  ka.t_part_max = t_part_max; ka.t_lse = teacher_lse;
  ka.part_max = part_max; ka.part_sum = part_sum;
  if (int rc = launch_kl_panel_emit<E>(ka, stream)) return rc;
  if (int rc = lse_from_partials(draft_hidden, draft_weight, hd, part_max, part_sum, draft_lse))
    return rc;
  {
    ScopedTimer timer(kClassCombine, stream);
    if (int rc = launch_kl_finish(losses, loss_part, tsum_part, pd.n_vtiles, pd.mp, draft_lse, m,
                                  stream))
      return rc;
  }
  KlGradFromExpArgs ga;
  ga.exp_panel = exp_panel; ga.teacher = teacher; ga.ld = pd.vp;
  ga.m = (int)m; ga.mp = (int)pd.mp;
  ga.part_max = part_max; ga.part_ld = (int)pd.mp; ga.draft_lse = draft_lse;
  ga.softcap = softcap;
  ga.t_part_max = t_part_max; ga.t_lse = teacher_lse;
  if (int rc = launch_kl_grad_from_exp(ga, pd.n_vtiles, stream)) return rc;

  if (int rc = prepare_k_tail(draft_weight, v, hd, ws + l.k_tail, stream)) return rc;
  GemmArgs g;
  set_head_operand(g, draft_weight, v, hd, ws + l.k_tail);
  g.b = exp_panel; g.ldb = pd.vp; g.b_rows = (int)pd.mp;
  g.k_per_split = 0;
  g.ni = fp.n_htiles; g.nj = (int)(pd.mp / E::kTile);
  g.c = slabs; g.ldc = hd; g.c_rows = (int)m; g.c_cols = (int)hd;
  g.c_split_stride = pd.mp * hd;
  g.mode = kStoreF32;
  if (int rc = launch_gemm<E, true, false>(g, fp.dh_ksplit, kClassGradHidden, stream)) return rc;
  ReduceSlabsArgs rs;
  rs.slabs = slabs; rs.n_splits = fp.dh_ksplit; rs.split_stride = pd.mp * hd;
  rs.row_scale = ones; rs.m = (int)m; rs.h = (int)hd;
  rs.out = unit_grad;
  return launch_reduce_slabs(rs, stream);
}

// Soft embedding without a usable soft cap (none, or one above kSoftEmbeddingMaxCap), in
// two contractions as well: one emitting pass over the head (entries relative to exact
// tile maxima, softmax partials), the lse merged from the partials with the embedding
// scale folded in, one elementwise pass that normalises the entries per (token, tile),
// and the contraction with the weight rows.
template <class E>
int soft_embedding_emit_impl(const FusedPlan& p, const void* hidden, const void* weight,
                             int64_t m, int64_t h, int64_t v, int dtype, float softcap,
                             float scale, void* out, char* ws, hipStream_t stream) {
  using T = typename E::T;
  const FusedLayout l = fused_layout(p, m, h, dtype, false);
  T* panel = reinterpret_cast<T*>(ws + l.panel);
  float* part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  float* part_max = reinterpret_cast<float*>(ws + l.part_max);
  float* lse = reinterpret_cast<float*>(ws + l.ref_next);
  float* row_scale = reinterpret_cast<float*>(ws + l.row_scale);
  float* slabs = reinterpret_cast<float*>(ws + l.slabs);
  const T* hidden_t = static_cast<const T*>(hidden);
  for (int block = 0; block < p.n_blocks; ++block) {
    const int64_t r0 = (int64_t)block * p.block_rows;
    const int64_t rows = std::min<int64_t>(p.block_rows, m - r0);
    if (rows <= 0) break;
    const int n_ttiles = (int)ceil_div(rows, E::kTile);
    const int64_t rows_p = (int64_t)n_ttiles * E::kTile;

    KlPanelArgs ka;
    ka.hidden = hidden_t + r0 * h; ka.weight = weight; ka.lse = nullptr; ka.scale = nullptr;
    ka.m = (int)rows; ka.h = (int)h; ka.v = (int)v; ka.softcap = softcap;
    ka.v0 = 0; ka.n_ttiles = n_ttiles; ka.n_ptiles = p.n_vtiles;
    ka.panel = panel; ka.ld = p.vp; ka.panel_in = nullptr;
    ka.loss_part = nullptr; ka.tsum_part = nullptr;
    ka.part_max = part_max; ka.part_sum = part_sum; ka.part_ld = (int)p.block_rows;
    ka.mode = kKlLoss;
    if (int rc = launch_kl_panel_emit<E>(ka, stream)) return rc;

    EmitRowsArgs er;
    er.part_max = part_max; er.part_sum = part_sum; er.part_ld = (int)p.block_rows;
    er.n_vtiles = p.n_vtiles; er.m = (int)rows; er.m_pad = (int)rows_p; er.scale = scale;
    er.lse = lse; er.row_scale = row_scale;
    if (int rc = launch_emit_rows(er, stream)) return rc;

    KlGradFromExpArgs ga;
    ga.exp_panel = panel; ga.teacher = nullptr; ga.ld = p.vp;
    ga.m = (int)rows; ga.mp = (int)rows_p;
    ga.part_max = part_max; ga.part_ld = (int)p.block_rows; ga.draft_lse = lse;
    ga.softcap = 0.0f;     // a forward value: no cap'
    if (int rc = launch_kl_grad_from_exp(ga, p.n_vtiles, stream)) return rc;

    GemmArgs g;
    set_head_operand(g, weight, v, h);
    g.b = panel; g.ldb = p.vp; g.b_rows = (int)rows_p;
    g.k_per_split = 0;
    g.ni = p.n_htiles; g.nj = n_ttiles;
    g.c = slabs; g.ldc = h; g.c_rows = (int)rows; g.c_cols = (int)h;
    g.c_split_stride = p.block_rows * h;
    g.mode = kStoreF32;
    const int ksplit = (rows_p == p.block_rows)
                           ? p.dh_ksplit
                           : std::min(p.dh_ksplit,
                                      grad_hidden_k_splits((int64_t)n_ttiles * p.n_htiles,
                                                           p.dh_ksplit, p.vp / 64, rows * h));
    if (int rc = launch_gemm<E, true, false>(g, ksplit, kClassGradHidden, stream)) return rc;
    ReduceSlabsArgs rs;
    rs.slabs = slabs; rs.n_splits = ksplit; rs.split_stride = p.block_rows * h;
    rs.row_scale = row_scale; rs.m = (int)rows; rs.h = (int)h;
    rs.out = nullptr; rs.out_t = static_cast<T*>(out) + r0 * h;
    if (int rc = launch_reduce_slabs(rs, stream)) return rc;
  }
  return 0;
}

#define TLCE_LAUNCHERS_EXP_GRADIENTS(X, E)                                              \
  X int launch_exp_panel_variant<E, false, false>(const ExpPanelArgs&, hipStream_t);    \
  X int launch_exp_panel_variant<E, true, false>(const ExpPanelArgs&, hipStream_t);
#define TLCE_LAUNCHERS_EXP_PANEL(X, E)                                                  \
  X int launch_kl_panel_emit<E>(const KlPanelArgs&, hipStream_t);                       \
  TLCE_LAUNCHERS_EXP_GRADIENTS(X, E)                                                    \
  X int launch_exp_panel_variant<E, true, true>(const ExpPanelArgs&, hipStream_t);      \
  X int launch_exp_panel_variant<E, false, false, true>(const ExpPanelArgs&, hipStream_t); \
  X int launch_exp_panel_variant<E, true, false, true>(const ExpPanelArgs&, hipStream_t);
#define TLCE_FUSED_GRADIENTS(X, E)                                                               \
  X int fused_gradients_impl<E>(const FusedPlan&, const void*, const void*, const int64_t*,      \
                                const int64_t*, int64_t, int64_t, int64_t, int, int64_t,         \
                                int64_t, float, float*, float*, float*, float*, float*, char*,   \
                                hipStream_t, const FusedOptions&);
#define TLCE_FUSED_ENTRY_POINTS(X, E)                                                            \
  TLCE_FUSED_GRADIENTS(X, E)                                                                     \
  X int soft_embedding_fused_impl<E>(const FusedPlan&, const void*, const void*, int64_t,        \
                                     int64_t, int64_t, int, float, float, void*, char*,          \
                                     hipStream_t);                                               \
  X int soft_embedding_emit_impl<E>(const FusedPlan&, const void*, const void*, int64_t,         \
                                    int64_t, int64_t, int, float, float, void*, char*,           \
                                    hipStream_t);                                                \
  X int topk_forward_with_gradient_impl<E>(const TopkPlan&, const FusedPlan&, const void*,       \
                                           const void*, const int64_t*, int64_t, int64_t,        \
                                           int64_t, int, float, float, float*, float*, float*,   \
                                           int64_t*, float*, float*, char*, hipStream_t);        \
  X int kl_forward_with_gradient_impl<E>(const Plan&, const Plan&, const KlLayout&,              \
                                         const FusedPlan&, const void*, const void*,             \
                                         const void*, const void*, int64_t, int64_t, int64_t,    \
                                         int64_t, int, float, float*, float*, float*, float*,    \
                                         char*, hipStream_t);                                    \
  X int deferred_contraction<E>(const FusedPlan&, const FusedLayout&, int64_t, int64_t, int64_t, \
                                const int64_t*, void*, char*, hipStream_t);                      \
  X int deferred_grad_weight_impl<E>(const FusedPlan&, const void*, int64_t, int64_t, int64_t,   \
                                     int, const float*, const float*, int, const int64_t*,       \
                                     const int64_t*, void*, char*, hipStream_t);

}  // namespace tlce
