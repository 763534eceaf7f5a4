// router.h -- a token's choice of experts (device code).
#pragma once
#include "device_util.h"
#include "moe.h"

namespace ffmi {

// wave-wide maximum on DPP (device library), the same in every lane
extern "C" __device__ float __ockl_wfred_max_f32(float);
// the wave's largest value, NV a lane (column i * 64 + lane; the lowest among equals).
// Picks follow one another, so a pick's latency counts: the maximum in the register
// file and a ballot for its place.  (Six steps of two shuffles through LDS: 38 tokens
// of 12 picks in one workgroup 17.2 us instead of 9.9.)
template <int NV>
__device__ __forceinline__ int best_column(const float (&v)[NV], float &best) {
  float m = v[0];
#pragma unroll
  for (int i = 1; i < NV; ++i) m = fmaxf(m, v[i]);
  best = __ockl_wfred_max_f32(m);
  int at = 0;
#pragma unroll
  for (int i = NV - 1; i >= 0; --i) {
    const unsigned long long where = __ballot(v[i] == best);
    if (where) at = i * 64 + __builtin_ctzll(where);
  }
  return at;
}
// A wave picks a token's experts: NV logits (z(column)) a lane, the best of the wave `top`
// times over.  A lane's pick, the lane-th of the token (-1: none).
template <int NV, class Z>
__device__ __forceinline__ int pick_experts(const Z &z, const float *__restrict__ bias, const MoeSizes &n,
                                            int t, const MoeLists &l) {
  const int lane = threadIdx.x & 63;
  const float gate = n.shared ? z(n.gate_col) : 0.f;
  float v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = i * 64 + lane;
    v[i] = -INFINITY;
    if (e < n.experts) {
      v[i] = z(e) + bias[e];
    }
  }
  float top0 = 0.f, sum = 0.f, mine = 0.f;  // lane k: the k-th pick
  int mine_e = 0;
  for (int k = 0; k < n.top; ++k) {
    float best;
    const int at = best_column<NV>(v, best);
    if (k == 0) top0 = best;
    const float p = expf(best - top0);
    sum += p;
    if (lane == k) mine = p, mine_e = at;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (at == i * 64 + lane) v[i] = -INFINITY;
  }
  if (lane < n.top) l.wt[(size_t)t * n.top + lane] = __fdiv_rn(mine, sum);
  if (n.shared && lane == 0) l.gate[t] = __fdiv_rn(1.0f, 1.0f + expf(-gate));
  return lane < n.top ? min(mine_e, n.experts - 1) : -1;
}
// the same by scores
template <int NV, class Z>
__device__ __forceinline__ int pick_experts(const Z &z, const MoeScores &sc, const MoeSizes &n, int t,
                                            const MoeLists &l) {
  const int lane = threadIdx.x & 63, cols = n.experts + n.identity, size = cols / sc.groups;
  float s[NV], v[NV];
  float mx = -INFINITY, sum = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = i * 64 + lane;
    s[i] = e < cols ? z(e) : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  mx = __ockl_wfred_max_f32(mx);
#pragma unroll
  for (int i = 0; i < NV; ++i) s[i] = expf(s[i] - mx), sum += s[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = i * 64 + lane;
    s[i] = __fdiv_rn(s[i], sum);
    v[i] = e < cols ? s[i] + sc.correction[e] : -INFINITY;
  }
  if (sc.keep < sc.groups) {  // the group of the best column left, `keep` times over
    float left[NV];
    bool in[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) left[i] = v[i], in[i] = false;
    for (int k = 0; k < sc.keep; ++k) {
      float best;
      const int g = best_column<NV>(left, best) / size;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if ((i * 64 + lane) / size == g) in[i] = true, left[i] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (!in[i]) v[i] = -INFINITY;
  }
  float mine = 0.f, total = 0.f, own = 0.f;
  int mine_e = 0;
  for (int k = 0; k < n.top; ++k) {
    float best, w = 0.f;
    const int at = best_column<NV>(v, best);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (at == i * 64 + lane) v[i] = -INFINITY, w = s[i];
    w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), at & 63));
    total += w;
    if (at >= n.experts) own += w;
    if (lane == k) mine = w, mine_e = at;
  }
  const float f = __fdiv_rn(sc.scale, total + 1e-20f);
  const bool real = lane < n.top && mine_e < n.experts;
  if (lane < n.top) l.wt[(size_t)t * n.top + lane] = real ? mine * f : 0.f;
  if (n.identity && lane == 0) l.own[t] = own * f;
  return real ? mine_e : -1;
}

// The router's product for one row, in the kernel that makes the row: the row in bf16 in
// LDS, the weights' 16 RT columns.  The sums are those of the product of few rows
// (gemm_skinny_kernel), bit for bit, so that a token's experts do not depend on how many
// tokens share its step: K in `slices`, each in kParts parts of consecutive k-steps, a part
// a chain of products; then the parts of a slice, then the slices, in order.  Wave w has
// slice w.  Its first kAhead k-steps of every part are fetched (begin) while the row is
// still being summed and normed (more than that: channels that 1024 does not divide).
template <int RT>
struct RouterRow {
  static constexpr int kParts = 4, kAhead = 2;
  h8 w[kParts][kAhead][RT];
  int kb, ke, per;
  // k-step j of part i, or none
  __device__ __forceinline__ bool has(int i, int j) const { return j < per && kb + i * per + j < ke; }
  __device__ __forceinline__ void load(const RouterWeights &r, int j0) {
    const uint16_t *p = r.w + (threadIdx.x & 63) * 8;
#pragma unroll
    for (int i = 0; i < kParts; ++i)
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        if (!has(i, j0 + j)) continue;
#pragma unroll
        for (int c = 0; c < RT; ++c)
          w[i][j][c] = *reinterpret_cast<const h8 *>(p + c * r.tile + (kb + i * per + j0 + j) * r.step);
      }
  }
  __device__ __forceinline__ void begin(const RouterWeights &r) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), mine = (r.steps + r.slices - 1) / r.slices;
    kb = wave < r.slices ? min(r.steps, wave * mine) : r.steps, ke = min(r.steps, kb + mine);
    per = (ke - kb + kParts - 1) / kParts;
    load(r, 0);
  }
  // row: the K values; sums [slices][16 RT] (barriers before and after are the caller's)
  __device__ __forceinline__ void product(const RouterWeights &r, const uint16_t *row, float *sums) {
    const int lane = threadIdx.x & 63;
    f4 acc[kParts][RT];
#pragma unroll
    for (int i = 0; i < kParts; ++i)
#pragma unroll
      for (int c = 0; c < RT; ++c) acc[i][c] = f4{0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < per; j0 += kAhead) {
      if (j0 > 0) load(r, j0);
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int i = 0; i < kParts; ++i) {
          if (!has(i, j0 + j)) continue;
          // (every column of 16 the same)
          const h8 x = *reinterpret_cast<const h8 *>(row + (kb + i * per + j0 + j) * 32 + 8 * (lane >> 4));
#pragma unroll
          for (int c = 0; c < RT; ++c)
            acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf8, w[i][j][c]), __builtin_bit_cast(bf8, x), acc[i][c], 0, 0, 0);
        }
    }
    const int wave = threadIdx.x >> 6;
    if ((lane & 15) || wave >= r.slices) return;
#pragma unroll
    for (int c = 0; c < RT; ++c)
      *reinterpret_cast<f4 *>(sums + wave * 16 * RT + c * 16 + (lane >> 4) * 4) =
          ((acc[0][c] + acc[1][c]) + acc[2][c]) + acc[3][c];
  }
};
template <int RT>
struct RouterTotal {
  const float *sums;
  int slices;
  __device__ __forceinline__ float operator()(int e) const {
    float v = sums[e];
    for (int i = 1; i < slices; ++i) v += sums[i * 16 * RT + e];
    return v;
  }
};

}  // namespace ffmi
