// Launch sequences of the float32 cross entropy on the bf16 matrix units
// (tlce_split_f32.h); their contractions are the kernels of tlce_kernels.h on SplitF32Engine.
#include "tlce_fused.h"
#include "tlce_split_f32.h"

namespace tlce {

TLCE_LAUNCHERS_FORWARD(extern template, SplitF32Engine)
TLCE_LAUNCHERS_GRAD_LOGITS(extern template, SplitF32Engine, false, false)
TLCE_LAUNCHERS_GRAD_LOGITS(extern template, SplitF32Engine, true, false)
TLCE_LAUNCHERS_GRAD_LOGITS(extern template, SplitF32Engine, false, true)
TLCE_LAUNCHERS_GRAD_LOGITS(extern template, SplitF32Engine, true, true)
extern template int launch_gemm<SplitF32Engine, true, false>(GemmArgs, int, int, hipStream_t);
extern template int launch_gemm<SplitF32Engine, true, true>(GemmArgs, int, int, hipStream_t);
TLCE_LAUNCHERS_EXP_GRADIENTS(extern template, SplitF32Engine)
TLCE_FUSED_GRADIENTS(template, SplitF32Engine)

// Eight columns per thread: 32 bytes in, 16 bytes per plane out.  Bound by memory.
__global__ __launch_bounds__(256) void lce_split_planes_kernel(const float* __restrict__ in,
                                                               int64_t rows, int64_t rows_pad,
                                                               int h, int hp,
                                                               __bf16* __restrict__ planes) {
  typedef __bf16 v8_t __attribute__((ext_vector_type(8)));
  const unsigned per_row = hp / 8;
  const int64_t pieces = rows_pad * per_row;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < pieces;
       i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / per_row;
    const int c = (int)(i - r * per_row) * 8;
    const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const float* src = in + r * h + c;
    const f32x4_t x0 =
        r < rows && c < h ? *reinterpret_cast<const f32x4_t*>(src) : zero;
    const f32x4_t x1 =
        r < rows && c + 4 < h ? *reinterpret_cast<const f32x4_t*>(src + 4) : zero;
    v8_t out[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float part[3];
      split_planes(e < 4 ? x0[e] : x1[e - 4], part);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) out[pl][e] = from_float<__bf16>(part[pl]);
    }
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
      *reinterpret_cast<v8_t*>(planes + (r * 3 + pl) * hp + c) = out[pl];
  }
}

int launch_split_planes(const float* in, int64_t rows, int64_t rows_pad, int64_t h, int64_t hp,
                        void* planes, hipStream_t stream) {
  const int64_t pieces = rows_pad * (hp / 8);
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(pieces, 256), 256 * 32));
  ScopedTimer timer(kClassTranspose, stream);
  lce_split_planes_kernel<<<grid, 256, 0, stream>>>(in, rows, rows_pad, (int)h, (int)hp,
                                                    static_cast<__bf16*>(planes));
  TLCE_LAUNCH_CHECK();
  return 0;
}

int split_forward(const SplitPlan& p, const void* hidden, const void* weight, const float* bias,
                  const int64_t* labels, const int64_t* row_idx, int64_t m, int64_t h, int64_t v,
                  int64_t ignore, int64_t exclude, float softcap, float* losses, float* lse,
                  float* valid_count, const ShardStats& shard, char* ws, hipStream_t stream,
                  const RowOptions& opt) {
  const SplitForwardLayout l =
      split_forward_layout(p, opt.weighted_sum != nullptr);
  float* part_max = reinterpret_cast<float*>(ws + l.part_max);
  float* part_sum = reinterpret_cast<float*>(ws + l.part_sum);
  if (int rc = launch_split_planes(static_cast<const float*>(hidden), m, p.mp, h, p.hp,
                                   ws + l.hidden, stream))
    return rc;
  for (int chunk = 0; chunk < p.n_chunks; ++chunk) {
    const int64_t v0 = (int64_t)chunk * p.chunk_tiles * 256;
    const int64_t rows = std::min<int64_t>((int64_t)p.chunk_tiles * 256, v - v0);
    if (int rc = launch_split_planes(static_cast<const float*>(weight) + v0 * h, rows, rows, h,
                                     p.hp, ws + l.weight, stream))
      return rc;
    ForwardArgs fa;
    fa.hidden = ws + l.hidden; fa.weight = ws + l.weight;
    fa.bias = bias != nullptr ? bias + v0 : nullptr;
    fa.m = (int)m; fa.h = (int)p.hp; fa.v = (int)rows;
    fa.exclude = exclude - shard.vocab_start - v0; fa.softcap = softcap;
    fa.logit_scale = opt.logit_scale;
    fa.n_ttiles = p.n_ttiles; fa.n_vtiles = (int)ceil_div(rows, 256); fa.nsplit = p.nsplit;
    fa.part_max = part_max + (int64_t)chunk * p.nsplit * p.mp;
    fa.part_sum = part_sum + (int64_t)chunk * p.nsplit * p.mp;
    fa.part_ld = (int)p.mp;
    Plan launch = {};
    launch.n_ttiles = p.n_ttiles; launch.n_vtiles = fa.n_vtiles; launch.nsplit = p.nsplit;
    if (int rc = launch_forward<SplitF32Engine>(launch, fa, stream)) return rc;
  }
  CombineArgs ca;
  ca.hidden = hidden; ca.weight = weight; ca.bias = bias; ca.labels = labels;
  ca.row_idx = row_idx;
  ca.m = (int)m; ca.h = (int)h; ca.v = (int)v;
  ca.ignore = ignore; ca.exclude = exclude; ca.softcap = softcap;
  ca.part_max = part_max; ca.part_sum = part_sum;
  ca.part_ld = (int)p.mp; ca.nsplit = p.n_chunks * p.nsplit;
  ca.losses = losses; ca.lse = lse; ca.valid_count = valid_count;
  return launch_combine<float>(ca, p.n_vtiles, 256, m, shard, ws + l.weighted, opt, stream);
}

int split_backward(const SplitPlan& p, const void* hidden, const void* weight, const float* bias,
                   const int64_t* labels, const int64_t* row_idx, const float* lse,
                   const float* valid_count, const float* grad_output, int64_t m, int64_t n_out,
                   int64_t h, int64_t v, int reduction, int64_t ignore, int64_t exclude,
                   float softcap, int64_t vocab_start, void* grad_hidden, void* grad_weight,
                   float* grad_bias, char* ws, hipStream_t stream, const RowOptions& opt) {
  const SplitBackwardLayout l = split_backward_layout(p, h);
  float* scale = reinterpret_cast<float*>(ws + l.scale);
  float* acc32 = reinterpret_cast<float*>(ws + l.acc32);
  ScaleArgs sa;
  sa.labels = labels; sa.row_idx = row_idx; sa.grad_output = grad_output;
  sa.valid_count = valid_count; sa.m = (int)m; sa.mp = (int)p.mp; sa.reduction = reduction;
  sa.ignore = ignore; sa.scale = scale; sa.constant = 0.0f;
  sa.multiplier = opt.logit_scale;
  sa.token_weights = opt.token_weights;
  if (int rc = launch_token_scale(sa, stream)) return rc;
  if (grad_bias != nullptr) {
    if (int rc = fill_zero(grad_bias, v * 4, stream)) return rc;
  }
  if (int rc = launch_split_planes(static_cast<const float*>(hidden), m, p.mp, h, p.hp,
                                   ws + l.hidden, stream))
    return rc;
  for (int panel = 0; panel < p.n_panels; ++panel) {
    const int64_t v0 = (int64_t)panel * p.vc;
    const int64_t width = std::min<int64_t>(p.vc, p.vp - v0);   // whole tiles
    const int64_t rows = std::min<int64_t>(p.vc, v - v0);       // real vocabulary rows
    if (int rc = launch_split_planes(static_cast<const float*>(weight) + v0 * h, rows, width, h,
                                     p.hp, ws + l.weight, stream))
      return rc;
    GradLogitsArgs ga;
    ga.hidden = ws + l.hidden; ga.weight = ws + l.weight;
    ga.bias = bias != nullptr ? bias + v0 : nullptr; ga.labels = labels;
    ga.lse = lse; ga.scale = scale;
    ga.m = (int)m; ga.h = (int)p.hp; ga.v = (int)rows;
    ga.ignore = ignore; ga.exclude = exclude - vocab_start - v0; ga.softcap = softcap;
    ga.label_offset = vocab_start + v0;
    ga.probabilities = 0; ga.cap_grad = 1;
    ga.logit_scale = opt.logit_scale;
    ga.v0 = 0;
    ga.n_ttiles = p.n_ttiles; ga.n_ptiles = (int)(width / 256);
    ga.g = ws + l.g; ga.ldg = p.vc; ga.gt = nullptr; ga.ldgt = 0;
    ga.grad_bias = bias != nullptr && grad_bias != nullptr ? grad_bias + v0 : nullptr;
    if (int rc = launch_grad_logits<SplitF32Engine>(ga, stream)) return rc;

    // grad_hidden: A = the planes of the panel's weight rows (K-major), B = G
    GemmArgs dh;
    dh.a = ws + l.weight; dh.lda = p.hp; dh.a_rows = (int)p.hp;
    dh.b = ws + l.g; dh.ldb = p.vc; dh.b_rows = (int)p.mp;
    dh.k = (int)round_up(rows, 64);
    dh.k_per_split = 0;
    dh.ni = p.n_htiles; dh.nj = p.n_ttiles;
    dh.c = acc32; dh.ldc = h; dh.c_rows = (int)m; dh.c_cols = (int)h;
    dh.c_split_stride = p.mp * h;
    dh.mode = panel == 0 ? kStoreF32 : kAddF32;
    if (int rc = launch_gemm<SplitF32Engine, true, false>(dh, p.dh_ksplit, kClassGradHidden, stream))
      return rc;
    if (grad_weight != nullptr) {
      // grad_weight: A = the planes of hidden, B = G, both K-major (K = token)
      GemmArgs dw;
      dw.a = ws + l.hidden; dw.lda = p.hp; dw.a_rows = (int)p.hp;
      dw.b = ws + l.g; dw.ldb = p.vc; dw.b_rows = (int)width;
      dw.k = (int)round_up(m, 64);
      dw.k_per_split = 0;
      dw.ni = p.n_htiles; dw.nj = (int)(width / 256);
      dw.c = static_cast<float*>(grad_weight) + v0 * h; dw.ldc = h;
      dw.c_rows = (int)rows; dw.c_cols = (int)h;
      dw.c_split_stride = 0;
      dw.mode = kStoreF32;
      if (int rc = launch_gemm<SplitF32Engine, true, true>(dw, 1, kClassGradWeight, stream)) return rc;
    }
  }
  if (row_idx != nullptr) {
    if (int rc = fill_zero(grad_hidden, n_out * h * 4, stream)) return rc;
  }
  ScopedTimer timer(kClassOther, stream);
  lce_finalize_grad_hidden_kernel<float><<<(int)m, 256, 0, stream>>>(
      acc32, p.dh_ksplit, p.mp * h, 0, row_idx, (int)m, (int)h, static_cast<float*>(grad_hidden),
      nullptr, p.n_htiles, 256, p.dh_ksplit, p.k_steps);
  TLCE_LAUNCH_CHECK();
  return 0;
}

}  // namespace tlce
