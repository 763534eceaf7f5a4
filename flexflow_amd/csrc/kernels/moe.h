// moe.h -- mixture of experts: routing, row lists, products by expert: launchers
// (moe.hip).
//
// A token's chosen experts are rows ("slots") of products grouped by expert: every
// expert's slots lie together, from a multiple of 16 on.  A shared expert that runs
// for every token joins the first product as one more group, its slots the tokens in
// order; its units, times the token's gate, are columns of a wider activation, so
// that its second product is part of a dense one.
#pragma once
#include "../ffmi_internal.h"

namespace ffmi {

struct MoeTile {
  int32_t expert;  // == number of experts: the shared one
  int32_t slot0, rows, pad;
};
constexpr int kMoeFew = 16, kMoeSome = 64, kMoeMany = 256;  // rows of a tile in the three forms
constexpr int kMoeMaxExperts = 1024, kMoeMaxTop = 64;

// a step's sizes: T tokens of which each takes `top` of `experts`
struct MoeSizes {
  int T = 0, experts = 0, top = 0;
  int identity = 0;  // further outputs of the router, after the experts': the row itself
  bool shared = false, f32 = false;
  int gate_col = 0;  // column of the shared expert's gate in the router's product
  // Few rows a tile: an expert's weights are read again for every 16 rows, on a large grid.
  // Many: once, on a grid that must not be small.  Some, between them: once for up to 64
  // rows, from registers.  Four layers' steps, us, of 4, 6, 8 and 11 rows an expert on
  // average, tokens all different, of 8 kinds and of 3, many and some:
  //   32 experts, 4 taken, 2752 x 4096  1639 1481  1725 1584  1728 1625  1790 1702
  //                                     1224 1087  1241 1134  1269 1182  1313 1294
  //                                      698  715   759  794   891  947   949 1049
  //   32, 4, 1408 x 2048                 618  545   656  595   691  624   721  664
  //                                      440  448   491  496   520  518   558  582
  //                                      406  345   447  389   472  446   507  493
  //   64, 8, 1024 x 2048                 726  669   772  720   833  786   871  835
  //                                      590  531   636  563   606  571   635  618
  //                                      439  438   464  471   504  554   534  590
  // (some loses where a handful of experts takes every row.  Tiles of 16 rows there instead:
  // 11 rows, 3 kinds 1408, 590, 641.)  From 14 rows on many is the faster.
  // A shared expert has every token's row: few read it T / 16 times (replay of 32 experts, 4
  // taken, and one of half the units, steps of 82 tokens: 18.3 ms, 19.0).
  // fp32 (16 rows a workgroup in any form): up to 12 rows an expert tiles of 16 spread them,
  // 32 experts, 704 x 2048, 48 tokens 4.9 -> 3.4 ms, 64 experts, 512 x 2048 6.2 -> 3.6.
  int tile_rows() const {
    if (T <= 32 || (long)T * top < 4L * experts) return kMoeFew;
    if (shared || (long)T * top >= 12L * experts) return kMoeMany;
    return f32 ? kMoeFew : kMoeSome;
  }
  // upper bounds: slots of the experts (whole 16s), tiles
  __host__ __device__ int slots() const {
    const int a = T * top, e = a < experts ? a : experts;
    return (a + 15 * e + 15) / 16 * 16;
  }
  int expert_tiles(int rows) const {
    const int a = T * top, e = a < experts ? a : experts;
    return (a - e) / rows + e;
  }
  __host__ __device__ int shared_tiles(int rows) const { return shared ? (T + rows - 1) / rows : 0; }
};
struct MoeLists {
  int32_t *picked = nullptr;      // [T][top] experts
  int32_t *at = nullptr;          // [T][top] slots (-1: none, an identity expert)
  float *wt = nullptr;            // [T][top] their weights
  float *gate = nullptr;          // [T] the shared expert's
  float *own = nullptr;           // [T] the identity experts' weights together
  int32_t *slot_token = nullptr;  // [slots]
  MoeTile *tiles = nullptr;       // the shared expert's first
  int32_t *num_tiles = nullptr;
};
// z: router products, the experts' columns first.  The `top` largest z + bias (the
// lowest index among equals), softmax over them; gate: the sigmoid of its column.
hipError_t launch_moe_route(const Partials &z, const float *bias, const MoeSizes &n, const MoeLists &l,
                            hipStream_t s);
// Another choice: scores s = softmax of all columns (identity experts' included); the
// `top` largest s + correction among the columns of the best `keep` of `groups` equal
// groups of neighbours (a group counts as its best column); weights scale s / (sum of
// the chosen s + 1e-20).
struct MoeScores {
  const float *correction = nullptr;  // [experts + identity]
  int groups = 1, keep = 1;
  float scale = 1.f;
};
hipError_t launch_moe_route_scores(const Partials &z, const MoeScores &sc, const MoeSizes &n, const MoeLists &l,
                                   hipStream_t s);
// The same in the kernel that makes a token's row: the product, the picks, their weights
// (MoeLists); the lists are then a launch of their own.
struct RouterWeights {
  const uint16_t *w = nullptr;  // bf16 packed, `steps` k-steps of 32 columns
  size_t tile = 0, step = 0;    // elements from tile to tile, k-step to k-step
  int steps = 0;
  int slices = 1;  // of K in the product of few rows (gemm_few_rows_slices), at most 8
};
struct RouteScores {
  RouterWeights w;
  MoeSizes n;
  MoeScores scores;
  MoeLists lists;
};
bool route_with_row(const MoeSizes &n, int H, int slices);  // (the rule) rows of H columns
hipError_t launch_moe_lists(const MoeSizes &n, const MoeLists &l, hipStream_t s);

// One product of every slot with its expert's matrix.
//   first  (gated): Y[slot] = silu(X W_gate) (X W_up), X the token's row (row-major),
//          Y bf16 in packed tiles of width ldy (fp32: rows); the shared expert's
//          times gate[token].  limit > 0: the clamped gated unit instead
//   second: Y[slot] = X W_down, X the first product's Y; Y rows of N, bf16 (fp32)
// W: bf16 packed weights, gate / up tiles in turn (fp32: rows, gate then up), expert
// after expert.
struct MoeGroup {
  const void *X = nullptr, *W = nullptr;
  void *Y = nullptr;
  int N = 0, K = 0, ldy = 0;
  size_t w_stride = 0;  // elements from expert to expert
};
struct MoeGemm {
  MoeGroup g[2];  // experts, shared (first product)
  int experts = 0;
  const int32_t *slot_token = nullptr;
  const MoeTile *tiles = nullptr;
  const int32_t *num_tiles = nullptr;
  const float *gate = nullptr;
  float limit = 0.f;
};
hipError_t launch_moe_gemm(const MoeGemm &a, const MoeSizes &n, bool gated, bool f32, bool stream_weights,
                           hipStream_t s);

}  // namespace ffmi
