// moe.hip -- mixture of experts (moe.h).
#include "moe.h"

#include <algorithm>

#include "device_util.h"
#include "router.h"

namespace ffmi {

// ---------------------------------------------------------------------------
// routing
// ---------------------------------------------------------------------------
// a column's sum over the slabs of a token's row, their loads together
struct SlabTotal {
  const float *row;
  size_t slab;
  int S;
  __device__ __forceinline__ SlabTotal(const Partials &z, int T, int t)
      : row(z.p + (size_t)t * z.NP), slab((size_t)T * z.NP), S(z.S) {}
  __device__ __forceinline__ float operator()(int e) const {
    float v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = row[e + min(s, S - 1) * slab];
#pragma unroll
    for (int s = 1; s < 8; ++s)
      if (s < S) v[0] += v[s];
    return v[0];
  }
};
// How: `const float *` (bias) or MoeScores
template <int NV, class How>
__global__ __launch_bounds__(256) void moe_pick_kernel(Partials z, How how, MoeSizes n, MoeLists l) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= n.T) return;
  const int e = pick_experts<NV>(SlabTotal(z, n.T, t), how, n, t, l);
  if (lane < n.top) l.picked[(size_t)t * n.top + lane] = e;
}

// first slot of every expert, from its count (a scan over the first wave), and the tiles
__device__ __forceinline__ void list_tiles(const int *count, int *next, const MoeSizes &n, const MoeLists &l,
                                           int rows) {
  const int tid = threadIdx.x, st = n.shared_tiles(rows);
  if (tid >= 64) {
    for (int i = tid - 64; i < st; i += 960)
      l.tiles[i] = MoeTile{n.experts, i * rows, min(rows, n.T - i * rows), 0};
    return;
  }
  const int per = (n.experts + 63) / 64, e0 = tid * per, e1 = min(e0 + per, n.experts);
  int slots = 0, tiles = 0;
  for (int e = e0; e < e1; ++e) slots += (count[e] + 15) & ~15, tiles += (count[e] + rows - 1) / rows;
  const int own_s = slots, own_t = tiles;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(slots, o), b = __shfl_up(tiles, o);
    if (tid >= o) slots += a, tiles += b;
  }
  if (tid == 63) *l.num_tiles = st + tiles;
  slots -= own_s, tiles += st - own_t;
  for (int e = e0; e < e1; ++e) {
    next[e] = slots;
    for (int r = 0; r < count[e]; r += rows)
      l.tiles[tiles++] = MoeTile{e, slots + r, min(rows, count[e] - r), 0};
    slots += (count[e] + 15) & ~15;
  }
}
// One workgroup: tokens by expert.  A pick's place among its expert's rows comes with
// the count.
//   NV > 0: it picks the experts as well, a token a wave (at most 16)
//   NV = 0: of picks made before, U a thread;  U = 0: of any number
template <int NV, int U, class How>
__global__ __launch_bounds__(1024) void moe_lists_kernel(Partials z, How how, MoeSizes n, MoeLists l,
                                                         int rows) {
  __shared__ int count[kMoeMaxExperts], next[kMoeMaxExperts];
  const int tid = threadIdx.x, A = n.T * n.top;
  for (int e = tid; e < n.experts; e += 1024) count[e] = 0;
  constexpr int R = U ? U : 1;
  int e[R], place[R];
  const int t = tid >> 6;
  if constexpr (NV) {
    e[0] = -1;
    if (t < n.T) e[0] = pick_experts<NV>(SlabTotal(z, n.T, t), how, n, t, l);
  } else if constexpr (U) {
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = tid + u * 1024 < A ? l.picked[tid + u * 1024] : -1;
  }
  __syncthreads();
  if constexpr (U) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e[u] >= 0) place[u] = atomicAdd(&count[e[u]], 1);
  } else {
    for (int a = tid; a < A; a += 1024)
      if (l.picked[a] >= 0) atomicAdd(&count[l.picked[a]], 1);
  }
  __syncthreads();
  list_tiles(count, next, n, l, rows);
  __syncthreads();
  const auto put = [&](int a, int token, int slot) {
    if (slot >= 0) l.slot_token[slot] = token;
    l.at[a] = slot;
  };
  if constexpr (NV) {
    const int lane = tid & 63;
    if (t < n.T && lane < n.top) put(t * n.top + lane, t, e[0] >= 0 ? next[e[0]] + place[0] : -1);
  } else if constexpr (U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int a = tid + u * 1024;
      if (a < A) put(a, a / n.top, e[u] >= 0 ? next[e[u]] + place[u] : -1);
    }
  } else {
    for (int a = tid; a < A; a += 1024) put(a, a / n.top, l.picked[a] >= 0 ? atomicAdd(&next[l.picked[a]], 1) : -1);
  }
}

// lists of picks made before
static void lists_of(const MoeSizes &n, const MoeLists &l, int rows, hipStream_t s) {
#define FFMI_ML(U)                                                                                              \
  hipLaunchKernelGGL((moe_lists_kernel<0, U, const float *>), dim3(1), dim3(1024), 0, s, Partials(), nullptr, n, l, \
                     rows)
  const long picks = (long)n.T * n.top;
  if (picks <= 1024) FFMI_ML(1);
  else if (picks <= 4096) FFMI_ML(4);
  else FFMI_ML(0);
#undef FFMI_ML
}
template <class How>
static hipError_t route(const Partials &z, How how, const MoeSizes &n, const MoeLists &l, hipStream_t s) {
  if (n.T <= 0) return hipSuccess;
  const int cols = n.experts + n.identity;
  if (n.experts < 1 || n.identity < 0 || cols > kMoeMaxExperts || n.top < 1 ||
      n.top > std::min(cols, kMoeMaxTop) || z.S < 1 || z.S > 8 || z.NP < cols ||
      (n.shared && n.gate_col >= z.NP) || (n.identity && !l.own))
    return hipErrorInvalidValue;
  const int rows = n.tile_rows();
  // Picks are vector instructions, 50 and more each: a workgroup's four SIMDs take as
  // long for 38 tokens (7.6 us, 4 of 32 experts; 50 for 64 tokens, 10 of 512) as the
  // workgroups of a launch before it would for hundreds (5.7; 13.6 both launches).  One
  // launch is the faster while a wave has one token (4.9 us for 16 tokens, 5.5 in two for
  // 17), with more than 64 columns or 16 picks up to about half the waves (128 columns, 8
  // picks: 5.1 for 8 tokens, 6.5 in two; 20 picks 10.6 for 16, 8.5 in two).
  const bool together = n.T <= (cols <= 64 && n.top <= 16 ? 16 : 8);
#define FFMI_ML(NV, U) \
  hipLaunchKernelGGL((moe_lists_kernel<NV, U, How>), dim3(1), dim3(1024), 0, s, z, how, n, l, rows)
#define FFMI_MR(NV)                                                                                          \
  do {                                                                                                       \
    if (together) {                                                                                          \
      FFMI_ML(NV, 1);                                                                                        \
    } else {                                                                                                 \
      hipLaunchKernelGGL((moe_pick_kernel<NV, How>), dim3((n.T + 3) / 4), dim3(256), 0, s, z, how, n, l);    \
      lists_of(n, l, rows, s);                                                                               \
    }                                                                                                        \
  } while (0)
  if (cols <= 64) FFMI_MR(1);
  else if (cols <= 128) FFMI_MR(2);
  else if (cols <= 256) FFMI_MR(4);
  else FFMI_MR(16);
#undef FFMI_MR
#undef FFMI_ML
  return hipGetLastError();
}
hipError_t launch_moe_lists(const MoeSizes &n, const MoeLists &l, hipStream_t s) {
  if (n.T <= 0) return hipSuccess;
  if (n.experts < 1 || n.identity < 0 || n.experts + n.identity > kMoeMaxExperts || n.top < 1 ||
      n.top > std::min(n.experts + n.identity, kMoeMaxTop))
    return hipErrorInvalidValue;
  lists_of(n, l, n.tile_rows(), s);
  return hipGetLastError();
}
hipError_t launch_moe_route(const Partials &z, const float *bias, const MoeSizes &n, const MoeLists &l,
                            hipStream_t s) {
  if (n.identity) return hipErrorInvalidValue;
  return route(z, bias, n, l, s);
}
hipError_t launch_moe_route_scores(const Partials &z, const MoeScores &sc, const MoeSizes &n, const MoeLists &l,
                                   hipStream_t s) {
  const int cols = n.experts + n.identity;
  if (sc.groups < 1 || cols % sc.groups || sc.keep < 1 || sc.keep > sc.groups ||
      n.top > cols / sc.groups * sc.keep || n.shared || !sc.correction)
    return hipErrorInvalidValue;
  return route(z, sc, n, l, s);
}

// ---------------------------------------------------------------------------
// products by expert
// ---------------------------------------------------------------------------
__device__ __forceinline__ f4 moe_mma(h8 a, h8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0,
                                                 0, 0);
}
__device__ __forceinline__ void store_bf16x4(uint16_t *p, float a, float b, float c, float d) {
  *reinterpret_cast<uint2 *>(p) =
      make_uint2(f2bf(a) | ((uint32_t)f2bf(b) << 16), f2bf(c) | ((uint32_t)f2bf(d) << 16));
}
// four consecutive output columns n.. of slot row m; gated: of the gate and up sums
// (f: the row's factor)
__device__ __forceinline__ float moe_unit(float gate, float up, float limit) {
  return limit > 0.f ? clamped_glu(gate, up, limit) : silu_glu(gate, up);
}
template <bool GATED>
__device__ __forceinline__ void moe_store(const MoeGroup &g, int m, int n, float f, float limit, const f4 &a,
                                          const f4 &b) {
  uint16_t *Y = (uint16_t *)g.Y;
  if constexpr (GATED)
    store_bf16x4(Y + act_packed_off(m, n, g.ldy), f * moe_unit(a[0], b[0], limit), f * moe_unit(a[1], b[1], limit),
                 f * moe_unit(a[2], b[2], limit), f * moe_unit(a[3], b[3], limit));
  else
    store_bf16x4(Y + (size_t)m * g.N + n, a[0], a[1], a[2], a[3]);
}

// Up to 16 rows: a workgroup has two 16-column tiles (a gate / up pair) and splits
// K over its four waves; weights straight to registers, U k-steps in flight.
template <bool GATED, bool NTL>
__global__ __launch_bounds__(256) void moe_few_kernel(MoeGemm a, int first, size_t wts) {
  constexpr int U = 8;
  __shared__ f4 red[3][2][64];
  if (first + (int)blockIdx.y >= *a.num_tiles) return;
  const MoeTile tl = a.tiles[first + blockIdx.y];
  const bool shared = tl.expert >= a.experts;
  const MoeGroup &g = a.g[shared];
  const int KT = g.K >> 5, ntiles = (GATED ? 2 : 1) * (g.N >> 4), tile0 = blockIdx.x * 2;
  if (tile0 >= ntiles) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m = lane & 15;
  const size_t wks = wts == 512 ? (size_t)ntiles * 512 : 512, ts = wts == 512 ? 512 : (size_t)KT * 512;
  const uint16_t *W = (const uint16_t *)g.W + (shared ? 0 : tl.expert * g.w_stride) + lane * 8;
  const uint16_t *w0 = W + tile0 * ts, *w1 = W + min(tile0 + 1, ntiles - 1) * ts;
  const uint16_t *x;
  if constexpr (GATED) {
    const int slot = tl.slot0 + min(m, tl.rows - 1);
    x = (const uint16_t *)g.X + (size_t)(shared ? slot : a.slot_token[slot]) * g.K + 8 * (lane >> 4);
  } else {
    x = (const uint16_t *)g.X + ((size_t)(tl.slot0 >> 4) * KT * 64 + packed_lane(lane, tl.rows)) * 8;
  }
  constexpr int XS = GATED ? 32 : 512;
  const int per = (KT + 3) / 4, kb = min(KT, wave * per), ke = min(KT, kb + per);
  f4 acc[2];
  acc[0] = acc[1] = f4{0.f, 0.f, 0.f, 0.f};
  const h8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = kb; k < ke; k += U) {
    h8 b[U][2], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t kk = min(k + u, ke - 1);
      b[u][0] = ld_weight<NTL>(w0 + kk * wks), b[u][1] = ld_weight<NTL>(w1 + kk * wks);
      xv[u] = *reinterpret_cast<const h8 *>(x + kk * XS);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= ke) xv[u] = zero;
      acc[0] = moe_mma(b[u][0], xv[u], acc[0]);  // D = W . X^T: a lane has 4 columns of a row
      acc[1] = moe_mma(b[u][1], xv[u], acc[1]);
    }
  }
  if (wave > 0) red[wave - 1][0][lane] = acc[0], red[wave - 1][1][lane] = acc[1];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < 3; ++w) acc[0] += red[w][0][lane], acc[1] += red[w][1][lane];
  if (m >= tl.rows) return;
  const int row = tl.slot0 + m, n = (lane >> 4) * 4;
  if constexpr (GATED) {
    moe_store<true>(g, row, blockIdx.x * 16 + n, shared ? a.gate[row] : 1.0f, a.limit, acc[0], acc[1]);
  } else {
    moe_store<false>(g, row, tile0 * 16 + n, 1.0f, 0.f, acc[0], acc[0]);
    if (tile0 + 1 < ntiles) moe_store<false>(g, row, tile0 * 16 + 16 + n, 1.0f, 0.f, acc[1], acc[1]);
  }
}

// The same of whole K and up to 64 rows, MT times 16: a wave has two tiles of its own, its
// sums in the tile kernel's order (a row's bits do not change where this form takes its
// place).  Two register sets: the next U k-steps are on their way while these are multiplied
// (with 64 rows U = 4 does not fit the registers of two waves a SIMD).
template <bool GATED, bool NTL, int MT, int U>
__device__ __forceinline__ void moe_chain(const MoeGemm &a, const MoeTile &tl, size_t wts) {
  const MoeGroup &g = a.g[0];
  const int lane = threadIdx.x & 63, m = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KT = g.K >> 5, ntiles = (GATED ? 2 : 1) * (g.N >> 4), pair = blockIdx.x * 4 + wave, tile0 = pair * 2;
  if (tile0 >= ntiles) return;
  const size_t wks = wts == 512 ? (size_t)ntiles * 512 : 512, ts = wts == 512 ? 512 : (size_t)KT * 512;
  const uint16_t *W = (const uint16_t *)g.W + tl.expert * g.w_stride + lane * 8;
  const uint16_t *w0 = W + tile0 * ts, *w1 = W + min(tile0 + 1, ntiles - 1) * ts;
  const uint16_t *x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r0 = min(i * 16, (tl.rows - 1) & ~15);  // (fewer rows than MT holds: the last 16 again)
    if constexpr (GATED)
      x[i] = (const uint16_t *)g.X + (size_t)a.slot_token[tl.slot0 + min(r0 + m, tl.rows - 1)] * g.K + 8 * (lane >> 4);
    else
      x[i] = (const uint16_t *)g.X + ((size_t)((tl.slot0 + r0) >> 4) * KT * 64 + packed_lane(lane, tl.rows - r0)) * 8;
  }
  constexpr int XS = GATED ? 32 : 512;
  f4 acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = f4{0.f, 0.f, 0.f, 0.f};
  h8 wa[U][2], xa[U][MT], wb[U][2], xb[U][MT];
  auto load = [&](h8(&b)[U][2], h8(&xv)[U][MT], int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t kk = min(k + u, KT - 1);
      b[u][0] = ld_weight<NTL>(w0 + kk * wks), b[u][1] = ld_weight<NTL>(w1 + kk * wks);
#pragma unroll
      for (int i = 0; i < MT; ++i) xv[u][i] = *reinterpret_cast<const h8 *>(x[i] + kk * XS);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mul = [&](const h8(&b)[U][2], const h8(&xv)[U][MT], int n) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u >= n) break;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        acc[i][0] = moe_mma(b[u][0], xv[u][i], acc[i][0]);
        acc[i][1] = moe_mma(b[u][1], xv[u][i], acc[i][1]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int k = 0;
  load(wa, xa, 0);
  for (; k + 2 * U < KT; k += 2 * U) {
    load(wb, xb, k + U);
    mul(wa, xa, U);
    load(wa, xa, k + 2 * U);
    mul(wb, xb, U);
  }
  if (k + U < KT) {
    load(wb, xb, k + U);
    mul(wa, xa, U);
    mul(wb, xb, KT - k - U);
  } else {
    mul(wa, xa, KT - k);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (i * 16 + m >= tl.rows) return;
    const int row = tl.slot0 + i * 16 + m, n = (lane >> 4) * 4;
    if constexpr (GATED) {
      moe_store<true>(g, row, pair * 16 + n, 1.0f, a.limit, acc[i][0], acc[i][1]);
    } else {
      moe_store<false>(g, row, tile0 * 16 + n, 1.0f, 0.f, acc[i][0], acc[i][0]);
      if (tile0 + 1 < ntiles) moe_store<false>(g, row, tile0 * 16 + 16 + n, 1.0f, 0.f, acc[i][1], acc[i][1]);
    }
  }
}
template <bool GATED, bool NTL>
__global__ __launch_bounds__(256, 2) void moe_chain_kernel(MoeGemm a, size_t wts) {
  if ((int)blockIdx.y >= *a.num_tiles) return;
  const MoeTile tl = a.tiles[blockIdx.y];
  if (tl.rows <= 16) moe_chain<GATED, NTL, 1, 8>(a, tl, wts);
  else if (tl.rows <= 32) moe_chain<GATED, NTL, 2, 4>(a, tl, wts);
  else moe_chain<GATED, NTL, 4, 2>(a, tl, wts);
}

// Up to 256 rows x 16 tiles a workgroup: eight waves as 2 (every other 16 rows) x 4
// (weight tiles); both operands' fragments go to LDS as they are stored (row-major
// rows: a lane fetches its own row's 16 bytes), NB - 1 k-steps in flight across raw
// barriers with counted waits, as the dense tile product does.  NF: 16-row fragments
// of a wave that hold rows; with up to 128 rows the other half is not fetched either.
template <bool GATED, int NF, int NB>
__device__ __forceinline__ void moe_tile(const MoeGemm &a, const MoeTile &tl, int tile0, size_t wts,
                                         h8 (*lds)[32][64]) {
  constexpr int OPS = NF > 4 ? 4 : 3;  // fragments that a wave fetches for a k-step
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool shared = tl.expert >= a.experts;
  const MoeGroup &g = a.g[shared];
  const int KT = g.K >> 5, ntiles = (GATED ? 2 : 1) * (g.N >> 4);
  const size_t wks = wts == 512 ? (size_t)ntiles * 512 : 512, ts = wts == 512 ? 512 : (size_t)KT * 512;
  const uint16_t *W = (const uint16_t *)g.W + (shared ? 0 : tl.expert * g.w_stride) + lane * 8;
  const uint16_t *src[OPS];
#pragma unroll
  for (int p = 0; p < OPS; ++p) {
    const int f = wave + 8 * p;
    if (p >= OPS - 2) {  // weight tiles
      src[p] = W + min(tile0 + f - 8 * (OPS - 2), ntiles - 1) * ts;
    } else if (GATED) {
      const int slot = tl.slot0 + min(f * 16 + (lane & 15), tl.rows - 1);
      src[p] = (const uint16_t *)g.X + (size_t)(shared ? slot : a.slot_token[slot]) * g.K + 8 * (lane >> 4);
    } else {
      const int mt = (tl.slot0 >> 4) + min(f, (tl.rows - 1) >> 4);
      src[p] = (const uint16_t *)g.X + ((size_t)mt * KT * 64 + lane) * 8;
    }
  }
  auto issue_one = [&](int kt, int p) {
    const bool w = p >= OPS - 2;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void *)(src[p] + (size_t)kt * (w ? wks : GATED ? 32 : 512)),
        (__attribute__((address_space(3))) void *)(&lds[kt % NB][wave + 8 * (w ? p - (OPS - 2) + 2 : p)][0]), 16,
        0, 0);
  };
  const int wm = wave >> 2, wn = wave & 3;
  f4 acc[NF][4];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < NB - 1; ++kt)
    if (kt < KT)
#pragma unroll
      for (int p = 0; p < OPS; ++p) issue_one(kt, p);
  static_assert(NB == 4, "the waits below count NB - 2 younger stages");
  for (int kt = 0; kt < KT; ++kt) {
    // step kt has arrived once at most the younger steps' loads remain; the barrier
    // makes every wave's visible and retires the reads of the buffer filled next
    const int ahead = min(KT - 1 - kt, NB - 2);
    if (ahead >= 2) {
      if constexpr (OPS == 4) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    } else if (ahead == 1) {
      if constexpr (OPS == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bool more = kt + NB - 1 < KT;
    const int buf = kt % NB;
    h8 xf[NF], wf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) wf[j] = lds[buf][16 + wn * 4 + j][lane];
#pragma unroll
    for (int i = 0; i < NF; ++i) xf[i] = lds[buf][2 * i + wm][lane];
#pragma unroll
    for (int i = 0; i < NF; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = moe_mma(wf[j], xf[i], acc[i][j]);
      if (more)
#pragma unroll
        for (int p = 0; p < OPS; ++p)  // (spread: a fetch's issue hides under the products)
          if (p * NF / OPS == i) issue_one(kt + NB - 1, p);
    }
  }
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int m = (2 * i + wm) * 16 + (lane & 15);
    if (m >= tl.rows) continue;
    const float f = GATED && shared ? a.gate[tl.slot0 + m] : 1.0f;
#pragma unroll
    for (int j = 0; j < 4; j += GATED ? 2 : 1) {
      const int tile = tile0 + wn * 4 + j;
      if (tile >= ntiles) continue;
      moe_store<GATED>(g, tl.slot0 + m, (GATED ? tile >> 1 : tile) * 16 + (lane >> 4) * 4, f, a.limit,
                       acc[i][j], acc[i][GATED ? j + 1 : j]);
    }
  }
}
// The shared expert's workgroups first (the longest), their row tiles of a column
// tile on one XCD; then the experts', a row tile's columns in turn.
template <bool GATED>
__global__ __launch_bounds__(512, 1) void moe_tile_kernel(MoeGemm a, int first, int st, int cols_shared,
                                                          int cols, size_t wts) {
  __shared__ __attribute__((aligned(1024))) h8 lds[4][32][64];
  const int nsh = st * cols_shared, b = blockIdx.x;
  int tile, col;
  if (b < nsh) {
    const int xcd = b & 7, q = nsh >> 3, r = nsh & 7;
    const int L = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (b >> 3);
    tile = L % st, col = L / st;
  } else {
    tile = first + st + (b - nsh) / cols, col = (b - nsh) % cols;
    if (tile >= *a.num_tiles) return;
  }
  const MoeTile tl = a.tiles[tile];
  const int frags = (tl.rows + 15) >> 4;
  if (frags <= 4) moe_tile<GATED, 2, 4>(a, tl, col * 16, wts, lds);
  else if (frags <= 8) moe_tile<GATED, 4, 4>(a, tl, col * 16, wts, lds);
  else if (frags <= 12) moe_tile<GATED, 6, 4>(a, tl, col * 16, wts, lds);
  else moe_tile<GATED, 8, 4>(a, tl, col * 16, wts, lds);
}

// fp32: 16 rows x 64 columns a workgroup
template <bool GATED>
__global__ __launch_bounds__(256) void moe_f32_kernel(MoeGemm a, int first) {
  __shared__ float sx[16][33], sw[GATED ? 2 : 1][64][33];
  if (first + (int)blockIdx.y >= *a.num_tiles) return;
  const MoeTile tl = a.tiles[first + blockIdx.y];
  const bool shared = tl.expert >= a.experts;
  const MoeGroup &g = a.g[shared];
  const int n0 = blockIdx.x * 64, tid = threadIdx.x, r = tid & 15, c = tid >> 4;
  if (n0 >= g.N) return;
  const float *W = (const float *)g.W + (shared ? 0 : tl.expert * g.w_stride);
  for (int m0 = 0; m0 < tl.rows; m0 += 16) {
    float acc[GATED ? 2 : 1][4];
#pragma unroll
    for (int p = 0; p < (GATED ? 2 : 1); ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[p][j] = 0.f;
    for (int k0 = 0; k0 < g.K; k0 += 32) {
      __syncthreads();
      for (int i = tid; i < 16 * 32; i += 256) {
        const int slot = tl.slot0 + min(m0 + i / 32, tl.rows - 1);
        sx[i / 32][i % 32] =
            ((const float *)g.X)[(size_t)(GATED && !shared ? a.slot_token[slot] : slot) * g.K + k0 + i % 32];
      }
#pragma unroll
      for (int p = 0; p < (GATED ? 2 : 1); ++p)
        for (int i = tid; i < 64 * 32; i += 256)
          sw[p][i / 32][i % 32] = W[((size_t)p * g.N + min(n0 + i / 32, g.N - 1)) * g.K + k0 + i % 32];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 32; ++k)
#pragma unroll
        for (int p = 0; p < (GATED ? 2 : 1); ++p)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[p][j] = fmaf(sx[r][k], sw[p][c + 16 * j][k], acc[p][j]);
    }
    if (m0 + r < tl.rows)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + c + 16 * j;
        const int row = tl.slot0 + m0 + r;
        if (n >= g.N) continue;
        if constexpr (GATED)
          ((float *)g.Y)[(size_t)row * g.ldy + n] =
              (shared ? a.gate[row] : 1.0f) * moe_unit(acc[0][j], acc[GATED ? 1 : 0][j], a.limit);
        else
          ((float *)g.Y)[(size_t)row * g.N + n] = acc[0][j];
      }
  }
}

hipError_t launch_moe_gemm(const MoeGemm &a, const MoeSizes &n, bool gated, bool f32, bool stream_weights,
                           hipStream_t s) {
  if (n.T <= 0) return hipSuccess;
  const bool shared = gated && n.shared;
  int N = 0;
  for (int i = 0; i < (shared ? 2 : 1); ++i) {
    const MoeGroup &g = a.g[i];
    if (g.N % 32 || g.K % 32 || g.N <= 0 || g.K <= 0 || (gated && (g.ldy < g.N || g.ldy % 32)))
      return hipErrorInvalidValue;
    N = std::max(N, g.N);
  }
  // (the second product leaves the shared expert's tiles out)
  const int rows = n.tile_rows(), st = shared ? n.shared_tiles(rows) : 0, first = n.shared_tiles(rows) - st;
  const int tiles = n.expert_tiles(rows);
  if (st + tiles > 65535 || (shared && !a.gate)) return hipErrorInvalidValue;
  if (f32) {
    const dim3 grid((N + 63) / 64, st + tiles);
    if (gated) hipLaunchKernelGGL(moe_f32_kernel<true>, grid, dim3(256), 0, s, a, first);
    else hipLaunchKernelGGL(moe_f32_kernel<false>, grid, dim3(256), 0, s, a, first);
    return hipGetLastError();
  }
  const int per = gated ? 2 : 1;
  const size_t wts = weights_kmajor() ? 512 : 0;
  if (rows == kMoeMany) {
    const int cols = (per * a.g[0].N / 16 + 15) / 16, cols_shared = st ? (per * a.g[1].N / 16 + 15) / 16 : 0;
    const dim3 grid(st * cols_shared + tiles * cols);
    if (gated)
      hipLaunchKernelGGL(moe_tile_kernel<true>, grid, dim3(512), 0, s, a, first, st, cols_shared, cols, wts);
    else
      hipLaunchKernelGGL(moe_tile_kernel<false>, grid, dim3(512), 0, s, a, first, st, cols_shared, cols, wts);
    return hipGetLastError();
  }
  const int pairs = (per * N / 16 + 1) / 2;
  const dim3 grid(pairs, st + tiles), quads((pairs + 3) / 4, tiles);
#define FFMI_MF(G, NL)                                                                            \
  do {                                                                                            \
    if (rows == kMoeSome) hipLaunchKernelGGL((moe_chain_kernel<G, NL>), quads, dim3(256), 0, s, a, wts); \
    else hipLaunchKernelGGL((moe_few_kernel<G, NL>), grid, dim3(256), 0, s, a, first, wts);       \
  } while (0)
  if (gated && stream_weights) FFMI_MF(true, true);
  else if (gated) FFMI_MF(true, false);
  else if (stream_weights) FFMI_MF(false, true);
  else FFMI_MF(false, false);
#undef FFMI_MF
  return hipGetLastError();
}

}  // namespace ffmi
