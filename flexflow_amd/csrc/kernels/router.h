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
// LDS, the weights' 16 RT columns split over NW waves by their k-steps.  A wave's first U
// k-steps are fetched (begin) while the row is still being summed and normed.
// Sums: of up to U / 4 k-steps, those of a wave, those of the waves, in order.
template <int RT, int NW>
struct RouterRow {
  static constexpr int U = 8;
  h8 w[U][RT];
  f4 acc[4][RT];
  int kb, ke;
  __device__ __forceinline__ void load(const RouterWeights &r, int k) {
    const uint16_t *p = r.w + (threadIdx.x & 63) * 8;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= ke) break;
#pragma unroll
      for (int j = 0; j < RT; ++j) w[u][j] = *reinterpret_cast<const h8 *>(p + j * r.tile + (k + u) * r.step);
    }
  }
  __device__ __forceinline__ void begin(const RouterWeights &r) {
    const int per = (r.steps + NW - 1) / NW;
    kb = min(r.steps, (int)(threadIdx.x >> 6) * per), ke = min(r.steps, kb + per);
    load(r, kb);
  }
  // row: the K values; sums [NW][16 RT] (barriers before and after are the caller's)
  __device__ __forceinline__ void product(const RouterWeights &r, const uint16_t *row, float *sums) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < RT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    for (int k = kb; k < ke; k += U) {
      if (k > kb) load(r, k);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k + u >= ke) break;
        const h8 x = *reinterpret_cast<const h8 *>(row + (k + u) * 32 + 8 * (lane >> 4));  // every column of 16 the same
#pragma unroll
        for (int j = 0; j < RT; ++j)
          acc[u / (U / 4)][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf8, w[u][j]), __builtin_bit_cast(bf8, x), acc[u / (U / 4)][j], 0, 0, 0);
      }
    }
    if (lane & 15) return;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const f4 v = ((acc[0][j] + acc[1][j]) + acc[2][j]) + acc[3][j];
      *reinterpret_cast<f4 *>(sums + (threadIdx.x >> 6) * 16 * RT + j * 16 + (lane >> 4) * 4) = v;
    }
  }
};
template <int RT, int NW>
struct RouterTotal {
  const float *sums;
  __device__ __forceinline__ float operator()(int e) const {
    float v = sums[e];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += sums[i * 16 * RT + e];
    return v;
  }
};

}  // namespace ffmi
