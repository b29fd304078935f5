// Float32 cross entropies on the bf16 matrix units: every float32 operand of a contraction
// is laid out once as three bf16 planes whose sum it is (split_planes: exact), and the
// direct-to-LDS engine runs its K loop six times, over the pairs of planes
//   lo.hi  hi.lo  mid.mid  mid.hi  hi.mid  hi.hi
// into the same float32 accumulators, smallest products first.  What is left out (mid.lo,
// lo.mid, lo.lo) is below 2^-24 of a product.
//
// What bounds the float32 engine is the float32 matrix rate, a sixteenth of bf16's; six
// bf16 passes take three eighths of the time at the nominal rates.  They are also the more
// exact: an MFMA adds 32 products to its accumulator at once where the float32 one adds
// four, so an eighth of the roundings at the sums' own magnitude (the other passes' sums
// are 2^-8 of it and less; largest first, the small products would be truncated against a
// full accumulator: 3 to 5 times the error, and a bias).
//
// Measured, float32 engine -> this, forward / forward and backward in us, and the 2-norm
// errors of loss, grad_hidden and grad_weight against float64:
//   1024 rows, H = 1024, V = 32000   618 / 2295 -> 414 / 1439  2.4e-7 1.2e-6 6.7e-7 -> 2.0e-7 3.3e-7 2.5e-7
//   2048 rows, H = 1024, V = 32000  1142 / 4446 -> 698 / 2621  2.4e-7 1.7e-6 8.9e-7 -> 2.0e-7 4.4e-7 3.2e-7
//   2048 rows, H = 2048, V = 50001  3448 / 13609 -> 2214 / 8497  2.3e-7 2.9e-6 9.0e-7 -> 1.9e-7 7.4e-7 3.2e-7
//    512 rows, H = 4096, V = 20000  1180 / 3453 -> 776 / 2246  4.9e-7 1.7e-6 1.1e-6 -> 2.3e-7 4.9e-7 4.0e-7
// of which laying out the planes of a 32000 x 1024 head takes 65 us, once per direction.
#pragma once

#include "tlce_host.h"

namespace tlce {

// planes[rows_pad][3][hp] of in[rows][h] (h a multiple of 4, hp of 64, h <= hp < h + 64): zero
// columns from h, zero rows from `rows` on.
int launch_split_planes(const float* in, int64_t rows, int64_t rows_pad, int64_t h, int64_t hp,
                        void* planes, hipStream_t stream);

// Bound of the planes of vocabulary rows that a launch reads (whole heads below it).
constexpr int64_t kSplitWeightBytes = 1ll << 30;

struct SplitPlan {
  int64_t hp;          // hidden size in whole K slabs
  int64_t mp, vp;
  int n_ttiles, n_vtiles, n_htiles;
  // forward: vocabulary chunks of chunk_tiles tiles (the last may be smaller), nsplit
  // vocabulary splits in each
  int chunk_tiles, n_chunks, nsplit;
  // backward: panels of vc vocabulary rows
  int64_t vc;
  int n_panels, dh_ksplit, dh_max_ksplit, k_steps;
};

// Where the six passes are the faster ones.  The float32 engine's tiles are a quarter of
// these 256x256 ones and need no planes, so small products stay with it; short K loops (small
// h) leave the epilogues, which split every logit gradient, as the larger part.
// Forward and backward, float32 engine / this, in us:
//   rows   256: H = 1024, V = 32000  685 / 761      384: 1027 / 815     512: 1213 / 864
//   rows   256: H = 2048, V = 50001 2128 / 1887     128: 1196 / 1689
//   tiles   64: 1024 rows, V = 4096, H = 1024  411 / 530, H = 4096  1305 / 1385
//          128: 2048 rows, V = 4096, H = 1024  676 / 669, H = 4096  2347 / 1659
//          128: 1024 rows, V = 8192, H = 1024  663 / 586;  512 rows, V = 16384, H = 512  390 / 387
//   vocabulary  1000: 8192 rows, H = 1024  1145 / 1359      2048: 1548 / 1466
//   hidden  256: 2048 rows, V = 32000  1244 / 1023, 8192 rows  4607 / 4777;  128: 725 / 821
//           512: 1024 rows, V = 16384   657 / 524
inline bool split_f32_supported(int64_t m, int64_t h, int64_t v, int dtype,
                                int64_t more_than_rows = 384, int64_t min_tiles = 128) {
  return dtype == TLCE_DTYPE_F32 && (h % 4) == 0 && h >= 512 && m > more_than_rows &&
         v >= 2048 && ceil_div(m, 256) * ceil_div(v, 256) >= min_tiles;
}

inline SplitPlan make_split_plan(int64_t m, int64_t h, int64_t v, int64_t panel_bytes) {
  SplitPlan p;
  constexpr int64_t tile = 256;
  p.hp = round_up(h, 64);
  p.mp = round_up(std::max<int64_t>(m, 1), tile);
  p.vp = round_up(v, tile);
  p.n_ttiles = (int)(p.mp / tile);
  p.n_vtiles = (int)(p.vp / tile);
  p.n_htiles = (int)ceil_div(h, tile);
  const int64_t plane_tile = p.hp * 6 * tile;   // bytes of one vocabulary tile's planes
  const int64_t most = std::max<int64_t>(1, kSplitWeightBytes / plane_tile);
  p.n_chunks = (int)ceil_div(p.n_vtiles, most);
  p.chunk_tiles = (int)ceil_div(p.n_vtiles, p.n_chunks);
  p.n_chunks = (int)ceil_div(p.n_vtiles, p.chunk_tiles);
  p.nsplit = forward_vocab_splits(p.n_ttiles, p.chunk_tiles, 256);
  if (panel_bytes <= 0) panel_bytes = kDefaultPanelBytes;
  int64_t tiles = std::max<int64_t>(1, std::min(panel_bytes / (p.mp * 6 * tile), most));
  p.n_panels = (int)ceil_div(p.n_vtiles, tiles);
  p.vc = ceil_div(p.n_vtiles, p.n_panels) * tile;
  p.n_panels = (int)ceil_div(p.vp, p.vc);
  // (a K step of the split rule is one of the K loop's, six per 64 vocabulary rows)
  p.k_steps = (int)(p.vc / 64) * SplitF32Engine::kPasses;
  p.dh_max_ksplit = (int)std::max<int64_t>(1, std::min<int64_t>(kMaxKSplits, p.vc / 64 / 2));
  p.dh_ksplit = grad_hidden_k_splits((int64_t)p.n_ttiles * p.n_htiles, p.dh_max_ksplit, p.k_steps,
                                     p.mp * h);
  return p;
}

struct SplitForwardLayout {
  int64_t hidden, weight, part_max, part_sum, weighted, total;
};
inline SplitForwardLayout split_forward_layout(const SplitPlan& p, bool dynamic_rows,
                                               bool weighted) {
  SplitForwardLayout l;
  int64_t off = 0;
  l.hidden = off;    off += align256(p.mp * p.hp * 6);
  l.weight = off;    off += align256((int64_t)p.chunk_tiles * 256 * p.hp * 6);
  int64_t floats = (int64_t)p.n_chunks * p.nsplit * p.mp;
  if (dynamic_rows) floats = std::max<int64_t>((int64_t)kTargetWorkgroups * 256, p.mp);
  l.part_max = off;  off += align256(floats * 4);
  l.part_sum = off;  off += align256(floats * 4);
  l.weighted = off;  off += weighted ? align256(p.mp * 4) : 0;
  l.total = off;
  return l;
}

struct SplitBackwardLayout {
  int64_t scale, acc32, hidden, weight, g, total;
};
inline SplitBackwardLayout split_backward_layout(const SplitPlan& p, int64_t h) {
  SplitBackwardLayout l;
  int64_t off = 0;
  l.scale = off;   off += align256(p.mp * 4);
  l.acc32 = off;   off += align256(p.mp * h * 4 * p.dh_ksplit);
  l.hidden = off;  off += align256(p.mp * p.hp * 6);
  l.weight = off;  off += align256(p.vc * p.hp * 6);
  l.g = off;       off += align256(p.mp * p.vc * 6);
  l.total = off;
  return l;
}

// Row counts kept on the device re-plan the vocabulary splits of one launch, so they take
// heads of one chunk.
inline bool split_forward_taken(int64_t m, int64_t h, int64_t v, int dtype, bool dynamic_rows) {
  return split_f32_supported(m, h, v, dtype) &&
         (!dynamic_rows || make_split_plan(m, h, v, 0).n_chunks == 1);
}

// The arguments are those of forward_impl / backward_impl (tlce_host.h), for float32.
int split_forward(const SplitPlan& p, const void* hidden, const void* weight, const float* bias,
                  const int64_t* labels, const int64_t* row_idx, int64_t m, int64_t h, int64_t v,
                  int64_t ignore, int64_t exclude, float softcap, float* losses, float* lse,
                  float* valid_count, const ShardStats& shard, char* ws, hipStream_t stream,
                  const RowOptions& opt);
int split_backward(const SplitPlan& p, const void* hidden, const void* weight, const float* bias,
                   const int64_t* labels, const int64_t* row_idx, const float* lse,
                   const float* valid_count, const float* grad_output, int64_t m, int64_t n_out,
                   int64_t h, int64_t v, int reduction, int64_t ignore, int64_t exclude,
                   float softcap, int64_t vocab_start, void* grad_hidden, void* grad_weight,
                   float* grad_bias, char* ws, hipStream_t stream, const RowOptions& opt);

}  // namespace tlce
