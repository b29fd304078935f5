// Row kernels of the forward that leaves the gradients (tlce_fused.h): the
// label-logit pass before the blocks, the per-block statistics / row-factor pass,
// the K-split reduction of grad_hidden and the final scale-and-cast.  Engine
// independent; compiled beside the C ABI.
#pragma once

#include "tlce_fused.h"

namespace tlce {

// One wave per row, 16 rows per workgroup; behind those, workgroups that count the rows with a
// loss (the first clears the flags), and workgroups that clear the losses and the map of rows.
// Those were launches of their own, as were the sum of the losses (now in the slab reduction)
// and the backward's two passes over rows and the clearing before them
// (lce_finish_rows_kernel): 5 us of host time each, which is what bounds small steps (64 rows
// over V = 32000 252 -> 224 us, 1036 rows 343 -> 322).
// One workgroup counts up to kRowsPerCount rows; more rows take several, which add to a count
// cleared by a launch before, and the losses' sum goes by parts likewise (kLossesPerBlock).  One
// workgroup for all was most of a step of many rows over few words: 2^20 rows, H = 64, V = 64,
// frozen, 3.40 ms, now 1.91; 262144 rows, H = 512, V = 256 1.25, now 0.91.
constexpr int kLabelRows = 16;
constexpr int kLabelThreads = 64 * kLabelRows;
constexpr int kClearPerBlock = 4096;
constexpr int kRowsPerCount = 16384;

template <typename T>
__global__ __launch_bounds__(kLabelThreads) void lce_label_logit_kernel(LabelLogitArgs p) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int extra = (int)blockIdx.x - (p.m + kLabelRows - 1) / kLabelRows;
  p.m = effective_rows(p.m, p.m_dev);
  if (extra >= 0 && extra < p.n_count) {
    __shared__ int sh_valid[kLabelRows];
    if (extra == 0) {
      for (int i = threadIdx.x; i < p.n_flags; i += kLabelThreads) p.flags[i] = 0;
    }
    const int last = (int)min((int64_t)p.m, (int64_t)(extra + 1) * kRowsPerCount);
    int valid = 0;
#pragma unroll 4
    for (int r = extra * kRowsPerCount + threadIdx.x; r < last; r += kLabelThreads)
      valid += p.labels[r] != p.ignore ? 1 : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) valid += __shfl_xor(valid, o, 64);
    if (lane == 0) sh_valid[wave] = valid;
    __syncthreads();
    if (threadIdx.x == 0) {
      int rows = 0;
#pragma unroll
      for (int w = 0; w < kLabelRows; ++w) rows += sh_valid[w];
      const float total = (float)rows;
      if (p.n_count == 1)
        p.valid_count[0] = total;
      else if (total != 0.0f)
        atomicAdd(p.valid_count, total);   // whole numbers: exact in any order
    }
    return;
  }
  if (extra >= p.n_count) {
    const int64_t first = (int64_t)(extra - p.n_count) * kClearPerBlock;
    const int64_t last = min(first + kClearPerBlock, p.n_out);
    for (int64_t i = first + threadIdx.x; i < last; i += kLabelThreads) {
      if (p.losses != nullptr) p.losses[i] = 0.0f;
      if (p.row_of != nullptr) p.row_of[i] = -1;
    }
    return;
  }
  const int r = blockIdx.x * kLabelRows + wave;
  if (r >= p.m) return;
  const int64_t label = p.labels[r];
  const bool valid = label != p.ignore;
  const bool here = valid && label >= 0 && label < p.v;
  float z = 0.0f;
  if (here) {
    const T* hrow = static_cast<const T*>(p.hidden) + (int64_t)r * p.h;
    const T* wrow = static_cast<const T*>(p.weight) + label * (int64_t)p.h;
    z = wave_dot<T>(hrow, wrow, p.h, lane) * p.logit_scale;
    if (p.softcap > 0.0f) z = p.softcap * tanhf(z / p.softcap);
  }
  if (lane == 0) {
    // a label on the excluded column or outside the vocabulary has no logit in the
    // loss (ce_forward_kernel, fused_linear_ce_cuda.cu:199-219); as a reference any
    // real column's logit serves
    p.target[r] = (here && label != p.exclude) ? z : 0.0f;
    p.ref[r] = valid ? z : INFINITY;
    if (p.row_map != nullptr) p.row_map[r] = valid ? r : -1;
  }
  if (sizeof(T) == 2 && p.rows_copy != nullptr) {
    typedef T v8_t __attribute__((ext_vector_type(8)));
    const v8_t zero = {};
    const T* from = static_cast<const T*>(p.hidden) + (int64_t)r * p.h;
    T* to = static_cast<T*>(p.rows_copy) + (int64_t)r * p.h;
    for (int k = lane * 8; k < p.h; k += 64 * 8)
      *reinterpret_cast<v8_t*>(to + k) =
          valid ? *reinterpret_cast<const v8_t*>(from + k) : zero;
  }
}

// 64 rows per workgroup of 16 waves, the rows across the lanes (coalesced: partials are
// stored [tile][row]).  Wave w adds the partials of the vocabulary tiles w, w + 16, ... in
// ascending order and the 16 sums are merged in wave order; then wave 0 finishes the 64
// rows, one per lane, and, when scaled_hidden is wanted, all waves write it, four rows each
// (rows past m only get their zero row of scaled_hidden and a zero row factor).  What
// bounds it is the latency of dependent loads: with 4 waves that finished 16 rows each, one
// after the other, 64 rows over 125 vocabulary tiles took 23 us (now 5), 1610 rows over 594
// tiles 84 us (now 13).
constexpr int kFusedRowsPerBlock = 64;
constexpr int kFusedRowsWaves = 16;

template <typename T>
__global__ __launch_bounds__(64 * kFusedRowsWaves) void lce_fused_rows_kernel(FusedRowsArgs p) {
  if (p.run_flag != nullptr && *p.run_flag == 0) return;
  if (p.m_dev != nullptr) {
    p.m = effective_block_rows(p.m, p.m_dev, p.row0);
    p.m_pad = min(p.m_pad, (p.m + 255) / 256 * 256);   // the token tiles the producer wrote
  }
  __shared__ float sh_sum[kFusedRowsWaves][kFusedRowsPerBlock];
  __shared__ float sh_max[kFusedRowsWaves][kFusedRowsPerBlock];
  __shared__ float sh_factor[kFusedRowsPerBlock];
  __shared__ float sh_entry[kFusedRowsWaves][kFusedRowsPerBlock];
  __shared__ float sh_rounded[kFusedRowsWaves][kFusedRowsPerBlock];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * kFusedRowsPerBlock;
  if (row0 >= p.m_pad) return;
  {
    const int r = row0 + lane;
    float sum = 0.0f, mx2 = -INFINITY;
    if (r < p.m) {
#pragma unroll 4
      for (int t = wave; t < p.n_vtiles; t += kFusedRowsWaves) {
        sum += p.part_sum[(int64_t)t * p.part_ld + r];
        mx2 = fmaxf(mx2, p.part_max[(int64_t)t * p.part_ld + r]);
      }
    }
    sh_sum[wave][lane] = sum;
    sh_max[wave][lane] = mx2;
    if (p.part_rounded != nullptr) {
      float entry = 0.0f, rounded = 0.0f;
      if (r < p.m) {
#pragma unroll 4
        for (int t = wave; t < p.n_vtiles; t += kFusedRowsWaves) {
          entry += p.part_entry[(int64_t)t * p.part_ld + r];
          rounded += p.part_rounded[(int64_t)t * p.part_ld + r];
        }
      }
      sh_entry[wave][lane] = entry;
      sh_rounded[wave][lane] = rounded;
    }
  }
  __syncthreads();
  if (wave == 0) {
    const int r = row0 + lane;
    float factor = 0.0f;
    if (r < p.m) {
      const float c = p.ref[r];
      const int64_t label = p.labels[r];
      // (by the label: a reference of +inf, what rows without loss carry, may also be a logit's)
      const bool live = label != p.ignore;
      float sum = sh_sum[0][lane], mx2 = sh_max[0][lane];
#pragma unroll
      for (int w = 1; w < kFusedRowsWaves; ++w) {
        sum += sh_sum[w][lane];
        mx2 = fmaxf(mx2, sh_max[w][lane]);
      }
      const float mx = mx2 * TLCE_LN2;
      const bool in_window = (mx - c <= p.window) && (mx - c >= -1.0f) && (sum > 0.0f) &&
                             (sum < 3.0e38f);
      const float target = p.target[r];
      const float w = (p.token_weights != nullptr) ? p.token_weights[r] : 1.0f;
      const float lse = live ? c + logf(sum) : 0.0f;
      if (live) factor = w * p.logit_scale / sum;
      if (p.part_rounded != nullptr) {
        float entry = sh_entry[0][lane], rounded = sh_rounded[0][lane];
#pragma unroll
        for (int q = 1; q < kFusedRowsWaves; ++q) {
          entry += sh_entry[q][lane];
          rounded += sh_rounded[q][lane];
        }
        if (live && rounded > 0.0f) factor *= entry / rounded;
        if (p.row_rounded != nullptr) {
          p.row_entry[r] = entry;
          p.row_rounded[r] = rounded;
        }
      }
      p.lse[r] = lse;
      const int64_t o = (p.row_idx != nullptr) ? p.row_idx[r] : p.loss_row0 + r;
      if (p.losses != nullptr) p.losses[o] = live ? lse - target : 0.0f;
      if (p.row_of != nullptr) p.row_of[o] = (int)(p.loss_row0 + r);
      if (p.probabilities != nullptr) p.probabilities[r] = live ? expf(target - lse) : 0.0f;
      p.ref_next[r] = (live && !in_window) ? mx : c;
      if (live && !in_window) atomicOr(p.redo, 1);
      float rest = 0.0f;
      // the label's entry: s * entry = (softmax - 1) * cap'
      if (!p.keep_label && live && label >= 0 && label < p.v && label != p.exclude) {
        float dcap = 1.0f;
        if (p.softcap > 0.0f) {
          const float t = target / p.softcap;
          dcap = 1.0f - t * t;
        }
        const float entry = (expf(target - c) - sum) * dcap;
        if constexpr (sizeof(T) == 4) {
          float part[3];
          split_planes(entry, part);
          __bf16* at = static_cast<__bf16*>(p.panel) + (int64_t)r * 3 * p.ld + label;
#pragma unroll
          for (int pl = 0; pl < 3; ++pl) at[pl * p.ld] = from_float<__bf16>(part[pl]);
        } else {
          const T rounded = from_float<T>(entry);
          static_cast<T*>(p.panel)[(int64_t)r * p.ld + label] = rounded;
          rest = entry - to_float<T>(rounded);
        }
      }
      if (p.label_rest != nullptr) p.label_rest[r] = rest;
    }
    if (r < p.m_pad) p.row_scale[r] = factor;
    sh_factor[lane] = factor;
  }
  T* scaled = static_cast<T*>(p.scaled_hidden);
  if (scaled == nullptr) return;
  __syncthreads();
  if constexpr (sizeof(T) == 4) {
    // float32: in planes of hp elements, zeros from h on (h a multiple of 4)
    for (int i = 0; i < kFusedRowsPerBlock / kFusedRowsWaves; ++i) {
      const int rr = wave * (kFusedRowsPerBlock / kFusedRowsWaves) + i;
      const int r = row0 + rr;
      if (r >= p.m_pad) return;
      const float factor = sh_factor[rr];
      const float* hrow = static_cast<const float*>(p.hidden) + (int64_t)min(r, p.m - 1) * p.h;
      __bf16* out = static_cast<__bf16*>(p.scaled_hidden) + (int64_t)r * 3 * p.hp;
      for (int k = lane * 4; k < p.hp; k += 64 * 4) {
        f32x4_t x = {0.0f, 0.0f, 0.0f, 0.0f};
        if (k < p.h && r < p.m) x = *reinterpret_cast<const f32x4_t*>(hrow + k);
        float part[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e) split_planes(x[e] * factor, part[e]);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          store4<__bf16>(out + pl * p.hp + k, part[0][pl], part[1][pl], part[2][pl], part[3][pl]);
      }
    }
    return;
  }
  for (int i = 0; i < kFusedRowsPerBlock / kFusedRowsWaves; ++i) {
    const int rr = wave * (kFusedRowsPerBlock / kFusedRowsWaves) + i;
    const int r = row0 + rr;
    if (r >= p.m_pad) return;
    const float factor = sh_factor[rr];
    const T* hrow = static_cast<const T*>(p.hidden) + (int64_t)min(r, p.m - 1) * p.h;
    T* out = scaled + (int64_t)r * p.h;
    if ((p.h % 8) == 0) {
      typedef T v8_t __attribute__((ext_vector_type(8)));
      for (int k = lane * 8; k < p.h; k += 64 * 8) {
        const v8_t x = *reinterpret_cast<const v8_t*>(hrow + k);
        v8_t y;
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = from_float<T>(to_float<T>(x[e]) * factor);
        *reinterpret_cast<v8_t*>(out + k) = y;
      }
    } else {
      for (int k = lane; k < p.h; k += 64) out[k] = from_float<T>(to_float<T>(hrow[k]) * factor);
    }
  }
}

__global__ __launch_bounds__(256) void lce_finish_rows_kernel(FinishRowsArgs p) {
  typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
  const int m = effective_rows(p.m, p.m_dev);
  const int64_t o = blockIdx.x;
  const v8_t zero = {};
  if (o >= p.n_out) {   // rows of the operand past the row count
    const int64_t r = (p.m_dev != nullptr ? 0 : p.m) + (o - p.n_out);
    if (r < m || r >= p.m_pad) return;
    v8_t* out = reinterpret_cast<v8_t*>(static_cast<__bf16*>(p.scaled) + r * p.h);
    for (int k = threadIdx.x; k < p.h / 8; k += 256) out[k] = zero;
    return;
  }
  const int64_t r = p.row_of != nullptr ? p.row_of[o] : o;
  v8_t* dst = reinterpret_cast<v8_t*>(static_cast<__bf16*>(p.grad_hidden) + o * p.h);
  if (r < 0 || r >= m) {
    for (int k = threadIdx.x; k < p.h / 8; k += 256) dst[k] = zero;
    if (p.holes && p.scaled != nullptr) {
      v8_t* out = reinterpret_cast<v8_t*>(static_cast<__bf16*>(p.scaled) + o * p.h);
      for (int k = threadIdx.x; k < p.h / 8; k += 256) out[k] = zero;
    }
    return;
  }
  float g = p.grad_output[p.reduction == TLCE_REDUCTION_NONE ? o : 0];
  if (p.reduction == TLCE_REDUCTION_MEAN) {
    // no row with a loss: every gradient entry is zero and stays zero
    const float count = p.valid_count[0];
    g = count > 0.0f ? g / count : 0.0f;
  }
  const float* src = p.grad_hidden32 + r * p.h;
  const bool operand = p.hidden != nullptr;
  const float factor = operand ? g * p.row_scale[r] : 0.0f;
  const __bf16* hrow = static_cast<const __bf16*>(p.hidden) + r * p.h;
  __bf16* scaled = static_cast<__bf16*>(p.scaled) + r * p.h;
  for (int k = threadIdx.x * 8; k < p.h; k += 256 * 8) {
    const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(src + k);
    const f32x4_t x1 = *reinterpret_cast<const f32x4_t*>(src + k + 4);
    v8_t y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = from_float<__bf16>((e < 4 ? x0[e] : x1[e - 4]) * g);
    dst[k / 8] = y;
    if (operand) {
      const v8_t x = *reinterpret_cast<const v8_t*>(hrow + k);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = from_float<__bf16>(to_float<__bf16>(x[e]) * factor);
      *reinterpret_cast<v8_t*>(scaled + k) = y;
    }
  }
}

// One wave per row, 16 rows per workgroup.
template <typename T>
__global__ __launch_bounds__(256) void lce_scale_rows_kernel(ScaleRowsArgs p) {
  float g = 0.0f;
  if (p.reduction != TLCE_REDUCTION_NONE) g = p.grad_output[0];
  if (p.reduction == TLCE_REDUCTION_MEAN) {
    const float count = p.valid_count[0];
    g = count > 0.0f ? g / count : 0.0f;
  }
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int m = effective_rows(p.m, p.m_dev);
  for (int i = 0; i < 4; ++i) {
    const int r = blockIdx.x * 16 + wave * 4 + i;
    if (r >= p.m_pad) return;
    if (p.reduction == TLCE_REDUCTION_NONE && r < m)
      g = p.grad_output[p.row_idx != nullptr ? p.row_idx[r] : (int64_t)r];
    const float factor = (r < m) ? g * p.row_scale[r] : 0.0f;
    const T* hrow = static_cast<const T*>(p.hidden) + (int64_t)min(r, max(m - 1, 0)) * p.h;
    T* out = static_cast<T*>(p.out) + (int64_t)r * p.h;
    typedef T v8_t __attribute__((ext_vector_type(8)));
    for (int k = lane * 8; k < p.h; k += 64 * 8) {
      v8_t y;
      if (r < m) {
        const v8_t x = *reinterpret_cast<const v8_t*>(hrow + k);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = from_float<T>(to_float<T>(x[e]) * factor);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = from_float<T>(0.0f);
      }
      *reinterpret_cast<v8_t*>(out + k) = y;
    }
  }
}

// Sum of the numbers from `first` up to `n` by one workgroup of 256 threads, in an order that
// depends on these alone.
template <class At>
__device__ __forceinline__ float block_sum(int64_t first, int64_t n, At&& at) {
  __shared__ float part[4];
  float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
  for (int64_t i = first + threadIdx.x; i < n; i += 1024) {
    s0 += at(i);
    if (i + 256 < n) s1 += at(i + 256);
    if (i + 512 < n) s2 += at(i + 512);
    if (i + 768 < n) s3 += at(i + 768);
  }
  const float s = wave_sum((s0 + s1) + (s2 + s3));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  return (part[0] + part[1]) + (part[2] + part[3]);
}

__global__ __launch_bounds__(256) void lce_sum_loss_parts_kernel(const float* parts, int n_parts,
                                                                 const float* valid_count,
                                                                 bool mean, float* loss) {
  const float sum = block_sum(0, n_parts, [&](int64_t i) { return parts[i]; });
  if (threadIdx.x == 0) loss[0] = mean ? sum / valid_count[0] : sum;
}

__global__ __launch_bounds__(256) void lce_reduce_scaled_slabs_kernel(ReduceSlabsArgs p) {
  const int r = blockIdx.x;
  if (p.loss != nullptr && r >= (int)gridDim.x - p.n_parts) {   // behind the rows
    const int part = r - ((int)gridDim.x - p.n_parts);
    const int64_t first = part * p.part_length;
    float sum;
    if (p.loss_weights == nullptr) {
      sum = block_sum(first, min(p.n_losses, first + p.part_length),
                      [&](int64_t i) { return p.losses[i]; });
    } else {
      const int64_t n = effective_rows((int)p.n_losses, p.m_dev);
      sum = block_sum(first, min(n, first + p.part_length), [&](int64_t i) {
        return p.loss_weights[i] * p.losses[p.loss_idx != nullptr ? p.loss_idx[i] : i];
      });
    }
    if (threadIdx.x != 0) return;
    if (p.n_parts > 1)
      p.loss_parts[part] = sum;
    else
      p.loss[0] = p.mean ? sum / p.valid_count[0] : sum;
    return;
  }
  if (p.m_dev != nullptr) {
    const int rows = effective_block_rows(p.m, p.m_dev, p.row0);
    if (r >= rows) return;
    p.n_splits = dynamic_k_splits(rows, true, p.n_htiles, p.tile, p.h, p.max_splits, p.slab_budget,
                                  p.k_steps, &p.split_stride);
  }
  const float s = p.row_scale[r];
  const float* src = p.slabs + (int64_t)r * p.h;
  // The label's entry, the softmax minus one, is nearly all of a row's gradient until the model
  // is certain, and so is its rounding to bf16: added back in float32, one row of the head read.
  float rest = 0.0f;
  const __bf16* label_row = nullptr;
  if (p.label_rest != nullptr) {
    rest = p.label_rest[r];
    label_row = static_cast<const __bf16*>(p.weight) + (rest != 0.0f ? p.labels[r] : 0) * p.h;
  }
  float fix[kTopkFix];
  const __bf16* fix_row[kTopkFix];
  if (p.fix_value != nullptr) {
#pragma unroll
    for (int j = 0; j < kTopkFix; ++j) {
      fix[j] = p.fix_value[(int64_t)r * kTopkFix + j];
      fix_row[j] = static_cast<const __bf16*>(p.weight) +
                   (int64_t)p.fix_id[(int64_t)r * kTopkFix + j] * p.h;
    }
  }
  typedef __bf16 v4_t __attribute__((ext_vector_type(4)));
  for (int k = threadIdx.x * 4; k < p.h; k += 256 * 4) {
    v4_t lw = {};
    if (label_row != nullptr) lw = *reinterpret_cast<const v4_t*>(label_row + k);
    f32x4_t sum = *reinterpret_cast<const f32x4_t*>(src + k);
#pragma unroll 8
    for (int q = 1; q < p.n_splits; ++q)
      sum += *reinterpret_cast<const f32x4_t*>(src + (int64_t)q * p.split_stride + k);
    if (rest != 0.0f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = fmaf(rest, to_float<__bf16>(lw[e]), sum[e]);
    }
    if (p.fix_value != nullptr) {
      v4_t w[kTopkFix];
#pragma unroll
      for (int j = 0; j < kTopkFix; ++j) w[j] = *reinterpret_cast<const v4_t*>(fix_row[j] + k);
#pragma unroll
      for (int j = 0; j < kTopkFix; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = fmaf(fix[j], to_float<__bf16>(w[j][e]), sum[e]);
    }
    sum = sum * s;
    if (p.out_t != nullptr) {
      store4<__bf16>(static_cast<__bf16*>(p.out_t) + (int64_t)r * p.h + k, sum[0], sum[1], sum[2],
                     sum[3]);
    } else {
      *reinterpret_cast<f32x4_t*>(p.out + (int64_t)r * p.h + k) = sum;
    }
  }
}

// blockIdx.x = row, blockIdx.y = a group of 8 vocabulary tiles: 32 threads per tile, 8
// columns each.  The logit gradient of the frozen-head KL from the two panels the
// forward left (rows from m on get zeros).
__global__ __launch_bounds__(256) void lce_kl_grad_from_exp_kernel(KlGradFromExpArgs p,
                                                                   int n_vtiles) {
  const int r = blockIdx.x;
  const int tile = blockIdx.y * 8 + (threadIdx.x >> 5);
  if (tile >= n_vtiles) return;
  const int64_t c = (int64_t)tile * 256 + (threadIdx.x & 31) * 8;
  __bf16* e = static_cast<__bf16*>(p.exp_panel) + (int64_t)r * p.ld + c;
  typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
  v8_t out;
  if (r < p.m && p.teacher == nullptr) {
    // only normalise: softmax (times what the caller folded into draft_lse)
    const float f = exp2f(p.part_max[(int64_t)tile * p.part_ld + r] -
                          p.draft_lse[r] * TLCE_LOG2E);
    const v8_t ev = *reinterpret_cast<const v8_t*>(e);
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = from_float<__bf16>(to_float<__bf16>(ev[i]) * f);
  } else if (r < p.m) {
    const float tile_max2 = p.part_max[(int64_t)tile * p.part_ld + r];
    const float f = exp2f(tile_max2 - p.draft_lse[r] * TLCE_LOG2E);
    const float ft = p.t_part_max != nullptr
                         ? exp2f(p.t_part_max[(int64_t)tile * p.part_ld + r] -
                                 p.t_lse[r] * TLCE_LOG2E)
                         : 1.0f;
    const float inv_cap = p.softcap > 0.0f ? TLCE_LN2 / p.softcap : 0.0f;
    const v8_t ev = *reinterpret_cast<const v8_t*>(e);
    const v8_t tv = *reinterpret_cast<const v8_t*>(static_cast<const __bf16*>(p.teacher) +
                                                   (int64_t)r * p.ld + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float ei = to_float<__bf16>(ev[i]);
      float g = ei * f - to_float<__bf16>(tv[i]) * ft;
      if (p.softcap > 0.0f) {
        // (an entry of 0 is a column past the vocabulary: its gradient is 0 anyway)
        const float t = ei > 0.0f ? (log2f(ei) + tile_max2) * inv_cap : 0.0f;
        g *= fmaxf(1.0f - t * t, 0.0f);   // (|z| <= cap: a rounded entry can say otherwise)
      }
      out[i] = from_float<__bf16>(g);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = from_float<__bf16>(0.0f);
  }
  *reinterpret_cast<v8_t*>(e) = out;
}

// Orders LDS accesses of one wave's lanes (its LDS instructions complete in order).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One wave per row, eight rows per workgroup (neighbouring rows' tile maxima share the 64-byte
// sectors they are read from); nothing is shared between the waves.  What bounds it is the
// latency of each row's chain: maxima, about k tiles of entries (512 bytes each), a few dot
// products of h.
constexpr int kSelectRows = 8;
constexpr int kSelectCap = 768;    // candidates; pruned beyond kSelectPrune (a tile adds 256)
constexpr int kSelectPrune = 512;

__global__ __launch_bounds__(64 * kSelectRows) void lce_topk_select_kernel(TopkSelectArgs p) {
  __shared__ unsigned ids_all[kSelectRows][kSelectCap];
  __shared__ unsigned short ent_all[kSelectRows][kSelectCap];   // bf16 bits of the entries
  // the tiles to read, then (in their place) the candidates' logits
  __shared__ float val_all[kSelectRows][kSelectPrune];
  __shared__ float fix_exact[kSelectRows][kTopkFix], fix_rounded[kSelectRows][kTopkFix];
  static_assert(kSelectPrune * sizeof(float) >= kTopkSelectTiles * sizeof(unsigned short), "");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = blockIdx.x * kSelectRows + wave;
  if (r >= p.m) return;
  unsigned* ids = ids_all[wave];
  unsigned short* ent = ent_all[wave];
  unsigned short* tiles = reinterpret_cast<unsigned short*>(val_all[wave]);
  float* val = val_all[wave];
  const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const __bf16* hrow = static_cast<const __bf16*>(p.hidden) + (int64_t)r * p.h;
  auto as_bf16 = [](unsigned bits) { return __uint_as_float(bits << 16); };

  // the row's tile maxima as keys that order like the numbers (NaN lowest: no tile holds one)
  constexpr int kKeys = kTopkSelectTiles / 64;
  unsigned key[kKeys];
  float row_max = -INFINITY;
#pragma unroll
  for (int i = 0; i < kKeys; ++i) {
    const int t = lane + 64 * i;
    key[i] = 0;
    if (t < p.n_vtiles) {
      const float mx = p.part_max[(int64_t)t * p.part_ld + r];
      const unsigned u = __float_as_uint(mx);
      key[i] = (u & 0x80000000u) ? ~u : u | 0x80000000u;
      row_max = fmaxf(row_max, mx);
    }
  }
  row_max = wave_max(row_max);
  // the k-th largest of them
  unsigned kth = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const unsigned trial = kth | (1u << bit);
    int count = 0;
#pragma unroll
    for (int i = 0; i < kKeys; ++i) count += __popcll(__ballot(key[i] >= trial));
    if (count >= p.k) kth = trial;
  }
  const float bound2 = __uint_as_float((kth & 0x80000000u) ? kth & 0x7fffffffu : ~kth);

  // every one of the k largest logits has an entry of at least `least`: their logits are at
  // least the bound, entries are rounded to bf16 (2^-9), and the logits of this pass and of
  // the dot products differ by float32 roundings.  Under a soft cap entries carry cap', which
  // lies between cap' at the bound and at the row's maximum.
  const float ref2 = (*p.redo != 0 ? p.ref_next[r] : p.ref[r]) * TLCE_LOG2E;
  const float slack2 = 0.02f + 1e-5f * fabsf(bound2);
  float dcap = 1.0f;
  if (p.softcap > 0.0f) {
    const float a = bound2 * TLCE_LN2 / p.softcap, b = row_max * TLCE_LN2 / p.softcap;
    dcap = fminf(1.0f - a * a, 1.0f - b * b);
  }
  const float down = dcap * exp2f(-slack2);
  float least = exp2f(bound2 - ref2) * down;
  // (entries stay normal numbers, and a factor near 0 would let everything in)
  bool settled = bound2 - ref2 > -100.0f && bound2 - ref2 < 100.0f && dcap > 0.05f;

  int count = 0;
  // the k-th largest entry so far (entries are not negative: their bits order like them)
  // raises `least`; what lies below it leaves the list
  auto prune = [&]() {
    wave_lds_order();
    unsigned top = 0;
    for (int bit = 14; bit >= 0; --bit) {
      const unsigned trial = top | (1u << bit);
      int n = 0;
      for (int i = 0; i < count; i += 64)
        n += __popcll(__ballot(i + lane < count && ent[i + lane] >= trial));
      if (n >= p.k) top = trial;
    }
    least = fmaxf(least, as_bf16(top) * down);
    int kept = 0;
    for (int i = 0; i < count; i += 64) {
      const bool in = i + lane < count;
      const unsigned id = in ? ids[i + lane] : 0;
      const unsigned e = in ? ent[i + lane] : 0;
      const bool keep = in && as_bf16(e) >= least;
      const unsigned long long mask = __ballot(keep);
      wave_lds_order();
      if (keep) {
        const int at = kept + __popcll(mask & below);
        ids[at] = id;
        ent[at] = (unsigned short)e;
      }
      kept += __popcll(mask);
      wave_lds_order();
    }
    count = kept;
  };
  if (settled) {
    int n_tiles = 0;
#pragma unroll
    for (int i = 0; i < kKeys; ++i) {
      const unsigned u = (key[i] & 0x80000000u) ? key[i] & 0x7fffffffu : ~key[i];
      const bool hit = key[i] != 0 && __uint_as_float(u) >= bound2 - slack2;
      const unsigned long long mask = __ballot(hit);
      if (hit) tiles[n_tiles + __popcll(mask & below)] = (unsigned short)(lane + 64 * i);
      n_tiles += __popcll(mask);
    }
    wave_lds_order();
    const __bf16* row = static_cast<const __bf16*>(p.panel) + (int64_t)r * p.ld;
    constexpr int kAhead = 8;   // tiles in flight
    for (int t0 = 0; t0 < n_tiles && settled; t0 += kAhead) {
      uint2 quad[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        quad[j] = *reinterpret_cast<const uint2*>(
            row + (int64_t)tiles[min(t0 + j, n_tiles - 1)] * 256 + lane * 4);
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        if (t0 + j >= n_tiles) break;
        const unsigned first = (unsigned)tiles[t0 + j] * 256 + lane * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const unsigned half = q < 2 ? quad[j].x : quad[j].y;
          const unsigned bits = (q & 1) ? half >> 16 : half & 0xffffu;
          const bool in = as_bf16(bits) >= least;
          const unsigned long long mask = __ballot(in);
          if (in) {
            const int at = count + __popcll(mask & below);
            ids[at] = first + q;
            ent[at] = (unsigned short)bits;
          }
          count += __popcll(mask);
        }
        if (count > kSelectPrune) {
          prune();
          if (count > kSelectPrune) {
            settled = false;
            break;
          }
        }
      }
    }
    if (settled) prune();
    settled = settled && count >= p.k && count <= min(3 * p.k + 96, kSelectPrune);
  }
  // (no correction until one is known; slots beyond k stay like this)
  if (lane < kTopkFix) {
    p.fix_value[(int64_t)r * kTopkFix + lane] = 0.0f;
    p.fix_id[(int64_t)r * kTopkFix + lane] = 0;
  }
  if (!settled) {
    // a row of zeros (padding): all logits are 0, the list is the first k words
    float any = 0.0f;
    for (int k = lane; k < p.h; k += 64) any = fmaxf(any, fabsf(to_float<__bf16>(hrow[k])));
    if (wave_max(any) == 0.0f && row_max == 0.0f) {
      for (int j = lane; j < p.k; j += 64) {
        p.top_values[(int64_t)r * p.k + j] = 0.0f;
        p.top_ids[(int64_t)r * p.k + j] = j;
      }
    } else if (lane == 0) {
      atomicOr(p.unsettled, 1);
    }
    return;
  }

  // the candidates' logits, four dot products at a time (each as wave_dot adds it up)
  bool numbers = true;
  typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
  for (int c = 0; c < count; c += 4) {
    const __bf16* w[4];
    float dot[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w[j] = static_cast<const __bf16*>(p.weight) + (int64_t)ids[min(c + j, count - 1)] * p.h;
      dot[j] = 0.0f;
    }
#pragma unroll 2
    for (int k = lane * 8; k < p.h; k += 64 * 8) {
      const v8_t a = *reinterpret_cast<const v8_t*>(hrow + k);
      v8_t b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const v8_t*>(w[j] + k);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          dot[j] = fmaf(to_float<__bf16>(a[e]), to_float<__bf16>(b[j][e]), dot[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float z = wave_sum(dot[j]) * p.logit_scale;
      if (p.softcap > 0.0f) z = p.softcap * tanhf(z / p.softcap);
      if (lane == 0 && c + j < count) val[c + j] = z;
      numbers = numbers && z == z;
    }
  }
  if (!numbers) {
    if (lane == 0) atomicOr(p.unsettled, 1);
    return;
  }
  wave_lds_order();
  // each by its rank: larger first, then the smaller id
  const int n_fix = min(p.k, kTopkFix);
  for (int i = lane; i < count; i += 64) {
    const float z = val[i];
    const unsigned id = ids[i];
    int rank = 0;
    for (int j = 0; j < count; ++j) {
      const float other = val[j];
      rank += (other > z || (other == z && ids[j] < id)) ? 1 : 0;
    }
    if (rank < p.k) {
      p.top_values[(int64_t)r * p.k + rank] = z;
      p.top_ids[(int64_t)r * p.k + rank] = id;
    }
    if (rank < n_fix) {
      float cap = 1.0f;
      if (p.softcap > 0.0f) {
        const float t = z / p.softcap;
        cap = 1.0f - t * t;
      }
      fix_exact[wave][rank] = exp2f(z * TLCE_LOG2E - ref2) * cap;
      fix_rounded[wave][rank] = as_bf16(ent[i]);
      p.fix_id[(int64_t)r * kTopkFix + rank] = (int)id;
    }
  }
  wave_lds_order();
  // The row factor came with entry / rounded in it, for the part of the rounding errors that all
  // entries share.  The fixed entries have none, so what they weigh must not enter: the others'
  // share alone is taken, and taken out of the fixed ones.  (With the label's word most of the
  // sum, its row of the head carried the error of the others' sum.)  Others below an eighth are
  // taken as they were rounded: their sum here is a difference, off by 1e-6 to 2e-6 of the whole,
  // and the error left in it about 1.5e-5 of itself.
  const float exact = wave_sum(lane < n_fix ? fix_exact[wave][lane] : 0.0f);
  const float stored = wave_sum(lane < n_fix ? fix_rounded[wave][lane] : 0.0f);
  const float entry = p.row_entry[r], rounded = p.row_rounded[r];
  const float others = rounded - stored;
  float common = 1.0f, sum = exact + others;
  if (others > 0.125f * rounded && fabsf((entry - exact) - others) < 0x1p-8f * others) {
    common = (entry - exact) / others;
    sum = entry;
  }
  if (lane < n_fix)
    p.fix_value[(int64_t)r * kTopkFix + lane] =
        fix_exact[wave][lane] / common - fix_rounded[wave][lane];
  if (lane == 0 && rounded > 0.0f && sum > 0.0f) p.row_scale[r] *= rounded / sum * common;
}

// One row and 2048 columns per workgroup, 8 columns per thread.
__global__ __launch_bounds__(256) void lce_exp_from_logits_kernel(ExpFromLogitsArgs p) {
  const int r = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= p.width) return;
  __bf16* dst = static_cast<__bf16*>(p.out) + (int64_t)r * p.ld_out + p.col0 + c;
  if (r >= p.m) {
    store4<__bf16>(dst, 0.0f, 0.0f, 0.0f, 0.0f);
    store4<__bf16>(dst + 4, 0.0f, 0.0f, 0.0f, 0.0f);
    return;
  }
  const float ref = p.run_max[r];
  if (c == 0) p.ref_used[r] = ref;
  const float* src = p.logits + (int64_t)r * p.ld + c;
  const f32x4_t z0 = *reinterpret_cast<const f32x4_t*>(src);
  const f32x4_t z1 = *reinterpret_cast<const f32x4_t*>(src + 4);
  float e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float z = i < 4 ? z0[i] : z1[i - 4];
    float x = __expf(z - ref);            // -inf (past the vocabulary) gives 0
    if (p.softcap > 0.0f) {
      const float t = z / p.softcap;
      x = (z > -INFINITY) ? x * (1.0f - t * t) : 0.0f;
    }
    e[i] = x;
  }
  store4<__bf16>(dst, e[0], e[1], e[2], e[3]);
  store4<__bf16>(dst + 4, e[4], e[5], e[6], e[7]);
}

// blockIdx.y = logits panel (all but the last, which was written with the final
// maxima): rows whose maximum grew after the panel was written are brought to the
// final reference.
__global__ __launch_bounds__(256) void lce_rescale_exp_rows_kernel(RescaleExpArgs p) {
  const int r = blockIdx.x;
  const int j = blockIdx.y;
  const float used = p.ref_used[(int64_t)j * p.m_pad + r];
  const float fin = p.run_max[r];
  if (used == fin) return;
  const float f = __expf(used - fin);
  const int64_t c0 = (int64_t)j * p.panel_width;
  const int64_t c1 = min(c0 + p.panel_width, p.total_width);
  __bf16* row = static_cast<__bf16*>(p.panel) + (int64_t)r * p.ld;
  typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
  for (int64_t c = c0 + threadIdx.x * 8; c < c1; c += 256 * 8) {
    v8_t x = *reinterpret_cast<v8_t*>(row + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = from_float<__bf16>(to_float<__bf16>(x[i]) * f);
    *reinterpret_cast<v8_t*>(row + c) = x;
  }
}

__global__ __launch_bounds__(256) void lce_topk_row_scale_kernel(TopkRowScaleArgs p) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= p.m_pad) return;
  p.row_scale[r] = (r < p.m) ? p.multiplier / p.run_sum[r] : 0.0f;
}

// One workgroup per row: grad_hidden[r, :] = ce_scale[r] * unit[r, :]
//   - ce_scale[r] * d'(label) * W[label] + sum_j grad_top_values[r, j] * d'(id_j) * W[id_j]
// (dflash_linear_topk.py:196-225) with d'(v) = multiplier * (1 - tanh^2(multiplier *
// h.W[v] / cap)) (multiplier alone without a cap), rounded once.  The coefficients
// of the single-row terms are formed first (under a soft cap one dot product each, a
// wave per entry), then every column is summed in float32.
constexpr int kTopkApplyMaxEntries = 257;   // top_k <= 256, plus the label

template <typename T>
__global__ __launch_bounds__(256) void lce_topk_apply_kernel(TopkApplyArgs p) {
  __shared__ float coef[kTopkApplyMaxEntries];
  __shared__ int64_t ids[kTopkApplyMaxEntries];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int r = blockIdx.x;
  const T* hrow = static_cast<const T*>(p.hidden) + (int64_t)r * p.h;
  const float scale = p.ce_scale[r];
  const int n_entries = (p.grad_top_values != nullptr ? p.k : 0) + 1;
  // one wave per entry, the waves taking every fourth: the raw logit is needed only for
  // the soft cap's derivative
  for (int e = wave; e < n_entries; e += 4) {
    const bool is_label = e == n_entries - 1;
    const int64_t id = is_label ? p.labels[r] : p.top_ids[(int64_t)r * p.k + e];
    const bool word = id >= 0 && id < p.v;
    const float weight_in = !word      ? 0.0f
                            : is_label ? -scale
                                       : p.grad_top_values[(int64_t)r * p.k + e];
    float deriv = p.logit_scale;
    if (p.softcap > 0.0f && weight_in != 0.0f) {   // wave-uniform
      const T* wrow = static_cast<const T*>(p.weight) + id * (int64_t)p.h;
      const float raw = wave_dot<T>(hrow, wrow, p.h, lane) * p.logit_scale;
      const float th = tanhf(raw / p.softcap);
      deriv *= 1.0f - th * th;
    }
    if (lane == 0) {
      coef[e] = weight_in * deriv;
      ids[e] = word ? id : 0;
    }
  }
  __syncthreads();
  // eight consecutive columns per thread and step (h is a multiple of 64 on this path):
  // 16-byte reads of the weight rows, 16-byte store
  const float* unit = p.unit + (int64_t)r * p.h;
  T* out = static_cast<T*>(p.grad_hidden) + (int64_t)r * p.h;
  typedef T v8_t __attribute__((ext_vector_type(8)));
  for (int k = t * 8; k < p.h; k += 256 * 8) {
    const f32x4_t u0 = *reinterpret_cast<const f32x4_t*>(unit + k);
    const f32x4_t u1 = *reinterpret_cast<const f32x4_t*>(unit + k + 4);
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = scale * (i < 4 ? u0[i] : u1[i - 4]);
    for (int e = 0; e < n_entries; ++e) {
      const float c = coef[e];
      if (c == 0.0f) continue;   // workgroup-uniform
      const v8_t w = *reinterpret_cast<const v8_t*>(static_cast<const T*>(p.weight) +
                                                    ids[e] * (int64_t)p.h + k);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = fmaf(c, to_float<T>(w[i]), acc[i]);
    }
    v8_t o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = from_float<T>(acc[i]);
    *reinterpret_cast<v8_t*>(out + k) = o;
  }
}

// 64 rows per workgroup of 16 waves, the rows across the lanes (the partials are
// stored [tile][row]: a wave reads 256 consecutive bytes per tile); wave w adds the
// tiles w, w + 16, ... in order and the 16 sums are merged in a fixed order.
constexpr int kSoftRowsWaves = 16;

__global__ __launch_bounds__(64 * kSoftRowsWaves) void lce_soft_rows_kernel(SoftRowsArgs p) {
  __shared__ float sh[kSoftRowsWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  float sum = 0.0f;
  if (r < p.m) {
    for (int t = wave; t < p.n_vtiles; t += kSoftRowsWaves)
      sum += p.part_sum[(int64_t)t * p.part_ld + r];
  }
  sh[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || r >= p.m_pad) return;
  sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kSoftRowsWaves; ++w) sum += sh[w][lane];
  p.row_scale[r] = (r < p.m && sum > 0.0f) ? p.scale / sum : 0.0f;
}

// The tiles' (maximum, sum) pairs of an emitting pass merged into lse - log(scale), the
// same way: 64 rows per workgroup of 16 waves, wave w merging the tiles w, w + 16, ...
// in ascending order, the 16 partial pairs merged in wave order.
__global__ __launch_bounds__(64 * kSoftRowsWaves) void lce_emit_rows_kernel(EmitRowsArgs p) {
  __shared__ float sh_max[kSoftRowsWaves][64];
  __shared__ float sh_sum[kSoftRowsWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  float mx = -INFINITY, sum = 0.0f;
  if (r < p.m) {
    for (int t = wave; t < p.n_vtiles; t += kSoftRowsWaves) {
      const float pm = p.part_max[(int64_t)t * p.part_ld + r];
      const float ps = p.part_sum[(int64_t)t * p.part_ld + r];
      if (pm > -INFINITY) {
        const float nm = fmaxf(mx, pm);
        sum = sum * exp2f(mx - nm) + ps * exp2f(pm - nm);   // (exp2f(-inf) = 0 the first time)
        mx = nm;
      }
    }
  }
  sh_max[wave][lane] = mx;
  sh_sum[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || r >= p.m_pad) return;
  if (r >= p.m) {
    p.lse[r] = 0.0f;
    p.row_scale[r] = 0.0f;
    return;
  }
  mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < kSoftRowsWaves; ++w) mx = fmaxf(mx, sh_max[w][lane]);
  sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kSoftRowsWaves; ++w)
    if (sh_max[w][lane] > -INFINITY) sum += sh_sum[w][lane] * exp2f(sh_max[w][lane] - mx);
  p.lse[r] = (mx + log2f(sum)) * TLCE_LN2 - logf(p.scale);
  p.row_scale[r] = 1.0f;
}

template <typename T>
__global__ __launch_bounds__(256) void lce_scale_cast_rows_kernel(ScaleCastArgs p) {
  const int64_t r = blockIdx.x;
  if (p.m_dev != nullptr && r >= *p.m_dev) return;
  const int64_t o = (p.row_idx != nullptr) ? p.row_idx[r] : r;
  float g = p.grad_output[p.reduction == TLCE_REDUCTION_NONE ? o : 0];
  if (p.reduction == TLCE_REDUCTION_MEAN) {
    // no row with a loss: every gradient entry is zero and stays zero
    const float count = p.valid_count[0];
    g = count > 0.0f ? g / count : 0.0f;
  }
  const float* src = p.in + r * p.h;
  T* dst = static_cast<T*>(p.out) + o * p.h;
  for (int k = threadIdx.x * 4; k < p.h; k += 256 * 4) {
    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(src + k);
    store4<T>(dst + k, x[0] * g, x[1] * g, x[2] * g, x[3] * g);
  }
}

}  // namespace tlce
