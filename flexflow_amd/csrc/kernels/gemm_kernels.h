// gemm_kernels.h -- skinny weight-streaming GEMM on MFMA for decode/verify shapes.
//
// Replaces the cublasGemmEx dense layer (linear_kernels.cu:450-582):
//   Y[T][N] = X[T][K] . W[N][K]^T, 16-bit in/out (fp16 or bf16), fp32 accumulate.
// (The reference runs cuBLAS with compute_type = fp16, linear_kernels.cu:509;
// accumulating in fp32 is a deliberate, documented precision upgrade.)
//
// Design (MI355X): at T <= ~200 the layer is HBM-bound on the weight stream
// (arithmetic intensity ~T flop/byte < the ~312 flop/byte ridge), so every
// weight byte must be read exactly once per step and at full bandwidth:
//  * weights are pre-packed in MFMA B-fragment order (weights.hip): a wave
//    streams contiguous 1 KiB per k-step, 16 B per lane, no LDS round trip
//    (guide: "GEMV / M <= 16: load straight to VGPRs, deep unroll");
//  * one workgroup owns NT 16-column tiles and splits K over its KW waves,
//    so small-N layers (o_proj, down_proj: 256 tiles) still put 8 waves on
//    every CU; U k-steps of loads are issued before their MFMAs;
//  * all M-tiles (<= MT*16 rows) of X share each weight fragment: weights
//    are read once regardless of T (X comes from L2);
//  * the per-element reduction order is fixed by (N-tile, K) only, so a
//    row's result does not depend on T or on which other rows are batched.
// Epilogue FFMI_EPI_SILU_MUL fuses SigmoidSiluMulti (sigmoid_silu_multi.cu:
// 37-47) on interleaved [gate|up] tiles.
// Included by gemm.hip (fp16) and gemm_bf16_*.hip, one translation unit per
// epilogue kind of the bf16 form.
#pragma once
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "../ffmi_internal.h"

namespace ffmi {

// compile-time loop: f(std::integral_constant<int, 0>) ... f(<N-1>)
template <int I, int N, class F>
__host__ __device__ __forceinline__ void static_for_impl(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_impl<I + 1, N>(f);
  }
}
template <int N, class F>
__host__ __device__ __forceinline__ void static_for(F &&f) {
  static_for_impl<0, N>(f);
}

// SigmoidSiluMultiKernel numerics (sigmoid_silu_multi.cu:41-46): gate and up
// are fp16 values, out = half(half(g * half(sigmoid(g))) * u)
__device__ __forceinline__ uint16_t silu_mul_h(float gacc, float uacc) {
  const float g = __half2float(__float2half_rn(gacc));
  const float u = __half2float(__float2half_rn(uacc));
  const float sg = __half2float(__float2half_rn(1.0f / (1.0f + expf(-g))));
  const float t = __half2float(__float2half_rn(g * sg));
  return __half_as_ushort(__float2half_rn(t * u));
}

// Epilogue kinds (the kernels' EPI parameter): the element type of X, W and Y
// goes with the kind, so one set of kernels serves both 16-bit formats.
//   0 fp16, plain     1 fp16, SiLU-mul of paired [gate|up] tiles
//   2 bf16, plain     3 bf16, squared ReLU     4 bf16 operands, fp32 slabs out
//   (4 always writes the split-K slab layout, S = 1 included: its consumer
//   takes the fp32 sums unrounded)
//   5 bf16, clamped gated unit of paired [gate|up] tiles (`lim`: its limit)
//   6 bf16, SiLU gate of paired [gate|up] tiles, fp32 up to the product
template <int EPI>
constexpr bool epi_bf16 = EPI >= 2;
template <int EPI>
constexpr bool epi_f32 = EPI == 4;
template <int EPI>
constexpr bool epi_paired = EPI == 1 || EPI == 5 || EPI == 6;
// (fragments are 16 raw bytes per lane in either format)
template <int EPI>
__device__ __forceinline__ f4 mma16(h8 a, h8 b, f4 c) {
  if constexpr (epi_bf16<EPI>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a),
                                                   __builtin_bit_cast(bf8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <int EPI>
__device__ __forceinline__ uint16_t out16(float v) {
  if constexpr (EPI == 3) {
    v = fmaxf(v, 0.f);
    v = v * v;
  }
  if constexpr (epi_bf16<EPI>) return f2bf(v);
  else return __half_as_ushort(__float2half_rn(v));
}

// output of a (gate, up) pair of sums
template <int EPI>
__device__ __forceinline__ uint16_t pair16(float g, float u, float lim) {
  if constexpr (EPI == 5) return f2bf(clamped_glu(g, u, lim));
  else if constexpr (EPI == 6) return f2bf(silu_glu(g, u));
  else return silu_mul_h(g, u);
}

// Split-K over workgroups (grid.y = S > 1, small-N layers only): each
// workgroup reduces its K slice over its waves and writes an fp32 partial
// slab [S][T][NTILES*16] that the consumer combines in slice order
// (Partials, the M-split kernel's slab layout).
// v of the lane n places further up the same 16-lane DPP row (row_ror:n)
template <int NR>
__device__ __forceinline__ float row_ror_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                               0x120 + NR, 0xf, 0xf, false));
}

// v of lane l (wave-uniform result), bit-exact
__device__ __forceinline__ float lane_f(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// The operand rows of a product behind a residual norm, made by every workgroup for
// itself (SumNormArgs): r = residual + half(sum of slabs), h = half(half(r * rms) * w),
// the norm kernel's arithmetic and order of sums (norm.hip: 128 threads a row).  The first
// workgroup of the grid stores r.  load() only asks for the two rows, so that the caller's
// weight loads go out behind it and their way hides the sums.
// Bound by latency: slabs, a barrier for the sum of squares and one for the rows, about
// 1.3 us more than the product alone, where the norm's launch took 3 and its boundary.  A
// model of 768 channels and 2 layers, 16 steps of one row 1434 -> 1381 us, of two 1484 ->
// 1416.  Three and four rows are two rounds of slabs in every workgroup: 1512 -> 1514 and 1517 ->
// 1526, so those keep their launches.
constexpr int kSumNormRows = 2;      // rows at most
constexpr int kSumNormWidth = 1024;  // columns at most
template <int MAXS>
struct SumNormRows {
  f4 lo[MAXS], hi[MAXS];
  uint4 x, w;
  __device__ __forceinline__ void load(const SumNormArgs &a, int T, int H) {
    const int row = min((int)(threadIdx.x >> 7), T - 1), ch = min((int)threadIdx.x & 127, (H >> 3) - 1);
    const float *q = a.sums + (size_t)row * a.NP + ch * 8;
#pragma unroll
    for (int s = 0; s < MAXS; ++s) {
      const float *qs = q + (size_t)min(s, a.S - 1) * T * a.NP;
      lo[s] = *reinterpret_cast<const f4 *>(qs);
      hi[s] = *reinterpret_cast<const f4 *>(qs + 4);
    }
    x = *reinterpret_cast<const uint4 *>(a.res_in + (size_t)row * H + ch * 8);
    w = *reinterpret_cast<const uint4 *>(a.wnorm + ch * 8);
  }
  // rows: LDS, complete behind the last barrier in here
  __device__ __forceinline__ void finish(const SumNormArgs &a, int T, int H,
                                         uint16_t (*rows)[kSumNormWidth + 8], bool store) {
    __shared__ double part[4];
    const int wave = threadIdx.x >> 6, row = threadIdx.x >> 7, ch = threadIdx.x & 127;
    const bool mine = ch < (H >> 3), real = mine && row < T;
#pragma unroll
    for (int s = 1; s < MAXS; ++s)
      if (s < a.S) lo[0] += lo[s], hi[0] += hi[s];
    union Row8 {
      uint4 v;
      _Float16 e[8];
    } r, wn, y;
    r.v = x, wn.v = w;
    double ss = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      r.e[q] = r.e[q] + (_Float16)(q < 4 ? lo[0][q] : hi[0][q - 4]);
      const float f = (float)r.e[q];
      if (mine) ss += (double)f * (double)f;
    }
    if (store && real) *reinterpret_cast<uint4 *>(a.res_out + (size_t)row * H + ch * 8) = r.v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    if ((threadIdx.x & 63) == 0) part[wave] = ss;
    __syncthreads();
    const float sum = (float)(part[wave & ~1] + part[wave | 1]);
    const float rms =
        (float)(_Float16)__fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)H), a.eps)));
#pragma unroll
    for (int q = 0; q < 8; ++q)
      y.e[q] = (_Float16)__fmul_rn((float)(_Float16)__fmul_rn((float)r.e[q], rms), (float)wn.e[q]);
    if (real) *reinterpret_cast<uint4 *>(&rows[row][ch * 8]) = y.v;
    __syncthreads();
  }
};

// FZ (FuseArgs, ffmi_internal.h): 1 = residual-add producer epilogue (EPI 0,
// unsplit), 2 = RMSNorm consumer prologue, 3 and 4 = the pair of an fp32 residual
// (EPI 4; EPI 4 and 5), 5 to 7 = rows made from slabs and residual in the prologue, of up
// to 8, 12 and 16 slabs (SumNormArgs; one row tile, KW 4).  Y is restrict-
// qualified except in the producer, where it aliases fz.res_in (the residual
// is updated in place).
template <int FZ>
using SkinnyY = std::conditional_t<FZ == 1, uint16_t *, uint16_t *__restrict__>;
// what a launch without norms carries of FuseArgs
struct PlainArgs {
  float limit;
};
template <int FZ>
using SkinnyArgs = std::conditional_t<FZ >= 5, SumNormArgs, std::conditional_t<FZ != 0, FuseArgs, PlainArgs>>;
template <int FZ>
constexpr int sum_norm_slabs = FZ == 5 ? 8 : FZ == 6 ? 12 : FZ == 7 ? 16 : 0;
template <int MT, int NT, int KW, int U, int EPI, bool PIPE = false, bool NTL = false, int FZ = 0>
__global__ __launch_bounds__(KW * 64) void gemm_skinny_kernel(
    const uint16_t *__restrict__ X, const uint16_t *__restrict__ Wp,
    SkinnyY<FZ> Y, float *__restrict__ Ypart, int T, int N, int K, int KT,
    int NTILES, int xp, int yp, size_t wts, size_t wks, SkinnyArgs<FZ> fz) {
  extern __shared__ __attribute__((aligned(16))) float red[];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // FZ >= 5: the rows' loads go out first, the sums wait for them behind the first weights'
  constexpr bool MAKE = FZ >= 5;
  static_assert(!MAKE || (MT == 1 && KW == 4 && !PIPE), "256 threads: two rows; a short K");
  __shared__ __attribute__((aligned(16))) uint16_t sRows[MAKE ? kSumNormRows : 1][MAKE ? kSumNormWidth + 8 : 8];
  SumNormRows<MAKE ? sum_norm_slabs<FZ> : 1> made;
  if constexpr (MAKE) made.load(fz, T, K);
  // FZ == 1: the residual this wave-0 epilogue adds, loaded up front
  _Float16 rpre[FZ == 1 ? MT : 1][FZ == 1 ? NT : 1][4];
  if constexpr (FZ == 1) {
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = min((int)(blockIdx.x * NT + j) * 16 + (lane & 15), N - 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = min(i * 16 + (lane >> 4) * 4 + r, T - 1);
            rpre[i][j][r] = reinterpret_cast<const _Float16 *>(fz.res_in)[(size_t)m * N + n];
          }
      }
    }
  }
  // FZ == 3: the residual and the norm weight of wave 0's epilogue
  float xpre[FZ == 3 ? MT : 1][FZ == 3 ? NT : 1][4], wpre3[FZ == 3 ? NT : 1];
  if constexpr (FZ == 3) {
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = min((int)(blockIdx.x * NT + j) * 16 + (lane & 15), N - 1);
        wpre3[j] = fz.w32 ? fz.w32[n] : 0.f;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            xpre[i][j][r] = fz.x[(size_t)min(i * 16 + (lane >> 4) * 4 + r, T - 1) * N + n];
      }
    }
  }
  // FZ == 2: rms of every row (the norm kernel's arithmetic on the
  // producer's per-tile sums of squares, summed in a fixed order), then the
  // rms of this lane's rows as an fp16 multiplier of its X fragments
  h8 rms8[FZ == 2 ? MT : 1];
  // wave w owns rows w, w + KW, ... (<= RPW of them); lane l sums partials
  // l, l + 64, ... (<= 4: nss <= 256) of each.  The loads go out first; the
  // sums, the LDS exchange and its barrier (rms_finish) run once the wave's
  // first batch of weight / X loads is in flight too (loads retire in order,
  // so waiting for these does not wait for those): the two round trips
  // overlap instead of adding up.  Every wave calls rms_finish exactly once.
  constexpr int RPW = (MT * 16 + KW - 1) / KW;
  constexpr bool RMS = FZ == 2 || FZ == 4;
  __shared__ float sRms[RMS ? MT * 16 : 1];
  float pv[RMS ? RPW : 1][4];
  // The norm weight comes once per workgroup and lies in LDS (8 KiB: K <= 4096).  A load of
  // its fragment per k-step, 64 bytes for 64 lanes, takes the L1 as long as one of X.
  // 12288 x 4096 and gate / up of 11008 x 4096, 8 rows: so and X in rows 20.6 and 31.3 us;
  // from LDS 19.0 and 29.9, X packed too 18.0 and 29.6; without a norm 17.1 and 28.9.
  constexpr int WPT = FZ == 2 ? 4096 / 8 / (KW * 64) : 1;
  __shared__ h8 sWn[FZ == 2 ? 4096 / 8 : 1];
  h8 wpre[WPT];
  bool rdone = FZ != 2 && !MAKE;
  if constexpr (FZ == 2) {
#pragma unroll
    for (int c = 0; c < WPT; ++c)
      wpre[c] = *reinterpret_cast<const h8 *>(fz.wnorm + (size_t)min((int)threadIdx.x + c * KW * 64, K / 8 - 1) * 8);
  }
  if constexpr (RMS) {
#pragma unroll
    for (int rr = 0; rr < RPW; ++rr) {
      const int m = min(wave + rr * KW, T - 1);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        pv[rr][c] = fz.ss_in[(size_t)m * fz.nss + min(lane + 64 * c, fz.nss - 1)];
    }
  }
  // a row's sum of squares: 16-lane DPP rows, then the four row sums in row order
  auto square_sum = [&](int rr) {
    float v = 0.f;
    if constexpr (RMS) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < fz.nss) v += pv[rr][c];
    }
    v += row_ror_f<1>(v);
    v += row_ror_f<2>(v);
    v += row_ror_f<4>(v);
    v += row_ror_f<8>(v);
    return ((lane_f(v, 0) + lane_f(v, 16)) + lane_f(v, 32)) + lane_f(v, 48);
  };
  // rms_finish contains the workgroup's only __syncthreads before the
  // cross-wave reduction.  It is called at several points (after the first
  // batch of loads of the pipelined loop, the batched loop or the tail, and
  // unconditionally after the k-loop) and runs once per wave (rdone): a wave
  // whose k-range is empty, or shorter than a batch, reaches it at the
  // post-loop call, so waves may arrive at s_barrier from different
  // program points.  That is well defined on CDNA (s_barrier counts waves,
  // not PCs); the builtin is convergent, so the compiler neither duplicates
  // nor moves it across the rdone branch.  Pinned by
  // test_gpu_kernels.py::test_fused_norm_consumer_empty_wave_ranges (KW 4 /
  // 8 with waves that own no k-step).
  auto rms_finish = [&]() {
    if constexpr (MAKE) {
      if (rdone) return;
      rdone = true;
      made.finish(fz, T, K, sRows, blockIdx.x == 0 && blockIdx.y == 0);
    }
    if constexpr (FZ == 2) {
      if (rdone) return;
      rdone = true;
#pragma unroll
      for (int c = 0; c < WPT; ++c) sWn[threadIdx.x + c * KW * 64] = wpre[c];
#pragma unroll
      for (int rr = 0; rr < RPW; ++rr) {
        const int m = wave + rr * KW;
        const float v = square_sum(rr);
        if (lane == 0 && m < T) {
          const float rf = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(v, (float)K), fz.eps)));
          sRms[m] = __half2float(__float2half_rn(rf));
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const _Float16 r = (_Float16)sRms[min(i * 16 + (lane & 15), T - 1)];
        rms8[i] = h8{r, r, r, r, r, r, r, r};
      }
    }
  };
  // norm weight fragment of k-step k (this lane's 8 columns)
  auto ldwn = [&](int k) -> h8 { return sWn[k * 4 + (lane >> 4)]; };
  // y = half(half(x * rms) * w): two fp16 multiplies, as the norm kernel
  auto nrm = [&](h8 &a, int i, const h8 &w) {
    if constexpr (FZ == 2) a = (a * rms8[i]) * w;
  };
  const int cb = blockIdx.x, ks = blockIdx.y, S = gridDim.y;
  const int tile0 = cb * NT;
  const int m0 = 0;
  const int per_wg = (KT + S - 1) / S;
  const int kb_wg = min(KT, ks * per_wg), ke_wg = min(KT, kb_wg + per_wg);
  const int per = (ke_wg - kb_wg + KW - 1) / KW;
  const int kb = min(ke_wg, kb_wg + wave * per);
  const int ke = min(ke_wg, kb + per);

  f4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};

  // X row-major, or packed activation tiles (xp): 1 KiB per fragment load
  const int XS = xp ? 512 : 32;
  const uint16_t *xrow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (xp) {
      const int mt = min((m0 + i * 16) >> 4, (T - 1) >> 4);
      xrow[i] = X + ((size_t)mt * KT * 64 + packed_lane(lane, T - mt * 16)) * 8;
    } else {
      const int r = min(m0 + i * 16 + (lane & 15), T - 1);
      xrow[i] = X + (size_t)r * K + 8 * (lane >> 4);
    }
  }
  // (FZ >= 5: from LDS, behind rms_finish)
  const uint16_t *made_row = &sRows[MAKE ? min(lane & 15, T - 1) : 0][MAKE ? 8 * (lane >> 4) : 0];
  const uint16_t *wrow[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int t = min(tile0 + j, NTILES - 1);
    wrow[j] = Wp + (size_t)t * wts + lane * 8;
  }

  int kt = kb;
  if constexpr (PIPE) {
    // software pipeline over batches of UP = U/2 k-steps, two register sets:
    // the next batch's loads are issued before this batch's MFMAs, so each
    // wave keeps UP..2*UP k-steps in flight
    constexpr int UP = U / 2;
    const int nb = (ke - kt) / UP;
    if (nb > 0) {
      h8 bA[UP][NT], aA[UP][MT], bB[UP][NT], aB[UP][MT];
      auto ld = [&](h8(&bb)[UP][NT], h8(&aa)[UP][MT], int k0) {
#pragma unroll
        for (int u = 0; u < UP; ++u)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            bb[u][j] = ld_weight<NTL>(wrow[j] + (size_t)(k0 + u) * wks);
#pragma unroll
        for (int u = 0; u < UP; ++u)
#pragma unroll
          for (int i = 0; i < MT; ++i)
            aa[u][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)(k0 + u) * XS);
      };
      auto mm = [&](h8(&bb)[UP][NT], h8(&aa)[UP][MT], int k0) {
        if constexpr (FZ == 2) {
          h8 ww[UP];
#pragma unroll
          for (int u = 0; u < UP; ++u) ww[u] = ldwn(k0 + u);
#pragma unroll
          for (int u = 0; u < UP; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i) nrm(aa[u][i], i, ww[u]);
        }
#pragma unroll
        for (int u = 0; u < UP; ++u)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
              acc[i][j] = mma16<EPI>(aa[u][i], bb[u][j], acc[i][j]);
      };
      ld(bA, aA, kt);
      rms_finish();
      int q = 0;
      for (; q + 2 < nb; q += 2) {
        ld(bB, aB, kt + UP);
        __builtin_amdgcn_sched_barrier(0);
        mm(bA, aA, kt);
        __builtin_amdgcn_sched_barrier(0);
        ld(bA, aA, kt + 2 * UP);
        __builtin_amdgcn_sched_barrier(0);
        mm(bB, aB, kt + UP);
        __builtin_amdgcn_sched_barrier(0);
        kt += 2 * UP;
      }
      if (q + 1 < nb) {  // two batches left
        ld(bB, aB, kt + UP);
        __builtin_amdgcn_sched_barrier(0);
        mm(bA, aA, kt);
        __builtin_amdgcn_sched_barrier(0);
        mm(bB, aB, kt + UP);
        kt += 2 * UP;
      } else {  // one batch left
        __builtin_amdgcn_sched_barrier(0);
        mm(bA, aA, kt);
        kt += UP;
      }
    }
  }
  for (; kt + U <= ke; kt += U) {
    h8 b[U][NT];
    h8 a[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        b[u][j] = ld_weight<NTL>(wrow[j] + (size_t)(kt + u) * wks);
    if constexpr (!MAKE)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          a[u][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)(kt + u) * XS);
    rms_finish();
    if constexpr (MAKE)
#pragma unroll
      for (int u = 0; u < U; ++u) a[u][0] = *reinterpret_cast<const h8 *>(made_row + (kt + u) * 32);
    // keep the whole batch of loads ahead of the MFMAs: left alone the
    // scheduler interleaves them and reuses registers, leaving ~7 loads in
    // flight per wave with a vmcnt wait before almost every MFMA
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FZ == 2)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const h8 wn = ldwn(kt + u);
#pragma unroll
        for (int i = 0; i < MT; ++i) nrm(a[u][i], i, wn);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mma16<EPI>(a[u][i], b[u][j], acc[i][j]);
  }
  // tail (< U k-steps; with a small K -- the SSM, K = 768 over 4-8 waves --
  // the whole loop): every load of the batch is issued before the first MFMA
  // (one memory round trip, not one per k-step).  Steps past ke re-load the
  // last step (valid addresses, no branch) and add a zero weight fragment.
  if (kt < ke) {
    const int rem = ke - kt;
    h8 b[U - 1][NT];
    h8 a[U - 1][MT];
#pragma unroll
    for (int u = 0; u < U - 1; ++u) {
      const int kk = min(kt + u, ke - 1);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        b[u][j] = ld_weight<NTL>(wrow[j] + (size_t)kk * wks);
      if constexpr (!MAKE)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          a[u][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)kk * XS);
    }
    rms_finish();
    if constexpr (MAKE)
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        a[u][0] = *reinterpret_cast<const h8 *>(made_row + min(kt + u, ke - 1) * 32);
    __builtin_amdgcn_sched_barrier(0);
    const h8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (FZ == 2)
#pragma unroll
      for (int u = 0; u < U - 1; ++u) {
        const h8 wn = ldwn(min(kt + u, ke - 1));
#pragma unroll
        for (int i = 0; i < MT; ++i) nrm(a[u][i], i, wn);
      }
#pragma unroll
    for (int u = 0; u < U - 1; ++u) {
      if (u >= rem)
#pragma unroll
        for (int j = 0; j < NT; ++j) b[u][j] = zero;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mma16<EPI>(a[u][i], b[u][j], acc[i][j]);
    }
  }

  rms_finish();  // (a wave with an empty k-range still meets the barrier)
  if constexpr (FZ == 4) {  // (read behind the reduction's barrier)
    static_assert(KW > 1, "");
#pragma unroll
    for (int rr = 0; rr < RPW; ++rr) {
      const int m = wave + rr * KW;
      const float v = square_sum(rr);
      if (lane == 0 && m < T) sRms[m] = __fdiv_rn(1.0f, sqrtf(__fdiv_rn(v, (float)fz.width) + fz.eps));
    }
  }
  // Cross-wave K reduction in a fixed order (wave 0 + 1 + ... + KW-1).
  if (KW > 1) {
    constexpr int REGS = MT * NT * 4;
    if (wave > 0) {
      float *dst = red + (size_t)(wave - 1) * REGS * 64;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) dst[((i * NT + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (wave != 0) return;
    for (int w = 1; w < KW; ++w) {
      const float *src = red + (size_t)(w - 1) * REGS * 64;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += src[((i * NT + j) * 4 + r) * 64 + lane];
    }
  }

  // Epilogue: C/D layout col = lane&15, row = (lane>>4)*4 + r.
  if constexpr (FZ == 3) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = (tile0 + j) * 16 + (lane & 15);
      const bool nok = tile0 + j < NTILES && n < N;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + i * 16 + (lane >> 4) * 4 + r;
          const float x = xpre[i][j][r] + acc[i][j][r];
          float sq = 0.f;
          if (nok && m < T) {
            fz.x[(size_t)m * N + n] = x;
            if (fz.w32) fz.hb[act_packed_off(m, n, N)] = f2bf(x * wpre3[j]);
            sq = x * x;
          }
          if (!fz.w32) continue;
          sq += row_ror_f<1>(sq);
          sq += row_ror_f<2>(sq);
          sq += row_ror_f<4>(sq);
          sq += row_ror_f<8>(sq);
          if ((lane & 15) == 0 && m < T && tile0 + j < NTILES) fz.ss_out[(size_t)m * NTILES + tile0 + j] = sq;
        }
    }
    return;
  }
  if constexpr (FZ == 4) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float f = sRms[min(m0 + i * 16 + (lane >> 4) * 4 + r, T - 1)];
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j][r] *= f;
      }
  }
  if (S > 1 || epi_f32<EPI>) {  // unpaired EPI only (host-checked)
    const int NP = NTILES * 16;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = (tile0 + j) * 16 + (lane & 15);
      if (tile0 + j >= NTILES) continue;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + i * 16 + (lane >> 4) * 4 + r;
          if (m < T) Ypart[((size_t)ks * T + m) * NP + n] = acc[i][j][r];
        }
    }
    return;
  }
  if constexpr (FZ == 1) {
    // residual add (the norm kernel's correctly rounded fp16 add of the
    // rounded GEMM output), then per (row, tile) the sum of squares of the
    // 16 new values: a fixed butterfly over the 16 lanes of the row
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = (tile0 + j) * 16 + (lane & 15);
      const bool nok = tile0 + j < NTILES && n < N;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + i * 16 + (lane >> 4) * 4 + r;
          const _Float16 rh = rpre[i][j][r] + (_Float16)acc[i][j][r];
          float sq = 0.f;
          if (nok && m < T) {
            reinterpret_cast<_Float16 *>(Y)[(size_t)m * N + n] = rh;
            if (fz.res_packed) reinterpret_cast<_Float16 *>(fz.res_packed)[act_packed_off(m, n, N)] = rh;
            const float f = (float)rh;
            sq = f * f;
          }
          // the 16 columns of the row are the 16 lanes of one DPP row:
          // rotate-and-add within the row (VALU, no LDS crossbar)
          sq += row_ror_f<1>(sq);
          sq += row_ror_f<2>(sq);
          sq += row_ror_f<4>(sq);
          sq += row_ror_f<8>(sq);
          if ((lane & 15) == 0 && m < T && tile0 + j < NTILES)
            fz.ss_out[(size_t)m * NTILES + tile0 + j] = sq;
        }
    }
    return;
  }
  if constexpr (!epi_paired<EPI>) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      int n = (tile0 + j) * 16 + (lane & 15);
      if (tile0 + j >= NTILES || n >= N) continue;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int m = m0 + i * 16 + (lane >> 4) * 4 + r;
          if (m < T)
            Y[yp ? act_packed_off(m, n, yp) : (size_t)m * N + n] = out16<EPI>(acc[i][j][r]);
        }
    }
  } else {
    // tiles (2p, 2p+1) = (gate, up) of output columns [16p, 16p+16)
    float lim = 0.f;
    if constexpr (!MAKE) lim = fz.limit;
    int n = cb * 16 + (lane & 15);
    if (n < N) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int m = m0 + i * 16 + (lane >> 4) * 4 + r;
          if (m >= T) continue;
          Y[yp ? act_packed_off(m, n, yp) : (size_t)m * N + n] =
              pair16<EPI>(acc[i][0][r], acc[i][1][r], lim);
        }
    }
  }
}

template <int MT, int NT, int KW, int U, int EPI, int FZ = 0>
static hipError_t run(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws, int T,
                      int N, int K, int KT, int NTILES, int S, hipStream_t s, int xp, int yp,
                      bool nt, int wpitch, const FuseArgs &fz = FuseArgs()) {
  const size_t wts = w_tile_stride(KT), wks = w_k_stride(wpitch);
  const int ncb = (NTILES + NT - 1) / NT;
  dim3 grid(ncb, S);
  size_t lds = KW > 1 ? (size_t)(KW - 1) * MT * NT * 4 * 64 * sizeof(float) : 0;
  // software-pipelined k-loop once every wave has >= 2 full batches (LLaMA-7B
  // decode at T = 8, cold: qkv 21.2 -> 19.5 us, gate/up 39.1 -> 36.8, lm_head
  // 49.5 -> 46.1); short loops (the SSM, K = 768) keep the batched form, which
  // the pipeline slowed (SSM lm_head warm 9.3 -> 12.1 us).
  // FFMI_SKINNY_PIPE=0/1 forces it off/on (A/B runs).
  static const int force = getenv("FFMI_SKINNY_PIPE") ? atoi(getenv("FFMI_SKINNY_PIPE")) : -1;
  const int per_wave = ((KT + S - 1) / S + KW - 1) / KW;
  const bool pipe = force >= 0 ? force != 0 : per_wave >= 2 * U;
  SkinnyArgs<FZ> args;
  if constexpr (FZ != 0) args = fz;
  else args.limit = fz.limit;
#define FFMI_SKINNY_LAUNCH(PP, NL)                                                             \
  hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, KW, U, EPI, PP, NL, FZ>), grid, dim3(KW * 64), \
                     lds, s, X, Wp, Y, ws, T, N, K, KT, NTILES, xp, yp, wts, wks, args)
  if (pipe) {
    if (nt) FFMI_SKINNY_LAUNCH(true, true);
    else FFMI_SKINNY_LAUNCH(true, false);
  } else {
    if (nt) FFMI_SKINNY_LAUNCH(false, true);
    else FFMI_SKINNY_LAUNCH(false, false);
  }
#undef FFMI_SKINNY_LAUNCH
  return hipGetLastError();
}

struct NoArgs {};
template <bool MAKE>
using WaveArgs = std::conditional_t<MAKE, SumNormArgs, NoArgs>;
// Wide, short-K layers (the 68M SSM's lm_head: 2000 tiles, K = 768): one
// WAVE per group of NT tiles over the whole K (a single MFMA chain per tile,
// no cross-wave reduction, no LDS), four independent waves per workgroup.
// The K-split form launches 1000 short 4-wave workgroups whose loads never
// fill the CU (13 us for 49 MB from the Infinity Cache); here each wave keeps
// two batches of UB k-steps in flight (double-buffered registers).
// MAKE: X's rows are made in the prologue (SumNormRows, up to 8 slabs), the wave's first
// weights asked for ahead of the sums.
template <int MT, int NT, int UB, bool NTL, int WPG = 4, int EPI = 0, bool MAKE = false>
__global__ __launch_bounds__(WPG * 64) void gemm_wave_kernel(const uint16_t *__restrict__ X,
                                                             const uint16_t *__restrict__ Wp,
                                                             uint16_t *__restrict__ Y,
                                                             float *__restrict__ Yf, int T, int N,
                                                             int KT, int NTILES, int xp, int yp,
                                                             size_t wts, size_t wks, WaveArgs<MAKE> a) {
  static_assert(!MAKE || (MT == 1 && WPG == 4), "256 threads: two rows");
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * WPG + (threadIdx.x >> 6);
  __shared__ __attribute__((aligned(16))) uint16_t sRows[MAKE ? kSumNormRows : 1][MAKE ? kSumNormWidth + 8 : 8];
  SumNormRows<MAKE ? 8 : 1> made;
  const uint16_t *made_row = &sRows[MAKE ? min(lane & 15, T - 1) : 0][MAKE ? 8 * (lane >> 4) : 0];
  if constexpr (MAKE) made.load(a, T, KT * 32);
  else if (g * NT >= NTILES) return;
  const int XS = xp ? 512 : 32;
  const uint16_t *xrow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (xp) {
      const int mt = min(i, (T - 1) >> 4);
      xrow[i] = X + ((size_t)mt * KT * 64 + packed_lane(lane, T - mt * 16)) * 8;
    } else {
      const int r = min(i * 16 + (lane & 15), T - 1);
      xrow[i] = X + (size_t)r * (KT * 32) + 8 * (lane >> 4);
    }
  }
  const uint16_t *wrow[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wrow[j] = Wp + (size_t)min(g * NT + j, NTILES - 1) * wts + lane * 8;
  f4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  h8 bA[UB][NT], xA[UB][MT], bB[UB][NT], xB[UB][MT];
  auto ld = [&](h8(&bb)[UB][NT], h8(&xx)[UB][MT], int k0) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int kk = min(k0 + u, KT - 1);
#pragma unroll
      for (int j = 0; j < NT; ++j) bb[u][j] = ld_weight<NTL>(wrow[j] + (size_t)kk * wks);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if constexpr (!MAKE) xx[u][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)kk * XS);
    }
  };
  const h8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  auto mm = [&](h8(&bb)[UB][NT], h8(&xx)[UB][MT], int k0) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      if constexpr (MAKE) xx[u][0] = *reinterpret_cast<const h8 *>(made_row + min(k0 + u, KT - 1) * 32);
      if (k0 + u >= KT) {  // past K: re-loaded fragments times a zero weight
#pragma unroll
        for (int j = 0; j < NT; ++j) bb[u][j] = zero;
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mma16<EPI>(xx[u][i], bb[u][j], acc[i][j]);
    }
  };
  ld(bA, xA, 0);
  if constexpr (MAKE) {
    made.finish(a, T, KT * 32, sRows, blockIdx.x == 0);
    if (g * NT >= NTILES) return;
  }
  for (int k0 = 0; k0 < KT; k0 += 2 * UB) {
    if (k0 + UB < KT) ld(bB, xB, k0 + UB);
    __builtin_amdgcn_sched_barrier(0);
    mm(bA, xA, k0);
    __builtin_amdgcn_sched_barrier(0);
    if (k0 + 2 * UB < KT) ld(bA, xA, k0 + 2 * UB);
    __builtin_amdgcn_sched_barrier(0);
    if (k0 + UB < KT) mm(bB, xB, k0 + UB);
    __builtin_amdgcn_sched_barrier(0);
  }
  // C layout: column lane & 15, rows (lane >> 4) * 4 + r
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = (g * NT + j) * 16 + (lane & 15);
    if (g * NT + j >= NTILES || n >= N) continue;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = i * 16 + (lane >> 4) * 4 + r;
        if (m >= T) continue;
        if constexpr (epi_f32<EPI>) Yf[(size_t)m * (NTILES * 16) + n] = acc[i][j][r];
        else Y[yp ? act_packed_off(m, n, yp) : (size_t)m * N + n] = out16<EPI>(acc[i][j][r]);
      }
  }
}

// Split-K factor of the skinny path, only where the consumer takes the partial
// slabs (no reduce pass).  Narrow layers (few column groups, e.g. the 68M SSM's
// o/down with 48 tiles) fill the chip by it.  From 128 tiles on: halves, where they even out
// what the busiest CU reads (a tile a workgroup: 384 tiles are two on half of the
// CUs, in halves three on each).  Cold, us, T = 4, 24 and 64: N 6144 x K 4096 11.6 -> 10.3, 15.6 -> 13.5,
// 23.2 -> 19.3; 4608 x 4096 10.6 -> 9.1, 14.5 -> 12.2, 22.7 -> 18.6; 6144 x 2048 7.5 -> 6.8, 9.6 -> 8.5, 14.1 ->
// 11.9; 2048 x 2048 4.7 -> 4.0, 6.2 -> 4.9, 8.8 -> 6.7; where they don't, at T = 8, 4096 x 4096 8.2 -> 8.8,
// 4096 x 11008 15.6 -> 16.1.  From 512 tiles on and more than 16 rows a workgroup takes two
// tiles (dispatch_nt), and the split is the same for all rows (a row's order of sums does not
// depend on how many there are), so both grids have to gain: 600 tiles, 9600 x 4096, 15.8 ->
// 14.3, 22.4 -> 19.1, 31.0 -> 25.1; but 786 tiles, 12576 x 4096, 20.1 -> 18.4, then 23.7 -> 24.6 and 31.9 ->
// 32.3, and 1376, 22016 x 4096, 29.9 -> 28.1, 33.6 -> 34.2, 45.7 -> 47.9 (two rounds and a half of
// two tiles are as good as three).  Nor what gemm_wave_kernel takes, whole K only: 22016 x 1024
// 10.4 -> 11.4, 12.2 -> 17.2, 17.4 -> 21.0.
// A tensor-parallel layer's column chunk is such a product too, its slabs summed by the
// all-reduce's copy-in (at most 1 MB more to read): 2048 x 1376 4.9 -> 3.7, 5.9 -> 4.5, 7.8 -> 6.0;
// 2048 x 2752 5.8 -> 5.3, 7.7 -> 6.4, 10.4 -> 8.0; 2048 x 5504 8.1 -> 6.5, 11.3 -> 8.5, 17.3 -> 10.8; 2048 x 1024
// 3.7 -> 3.6, 4.6 -> 4.3, 6.4 -> 5.2.
// Four slices gain little more (6144 x 4096 9.9, 6144 x 2048 6.5) and cost a
// consumer that reads every sum several times (matrix memories) more than that.
// A wave keeps 4 k-steps or more.
static int skinny_split(int T, int N, int K, int epi, bool deferrable) {
  // FFMI_SKINNY_SPLIT=0 keeps every skinny launch unsplit (A/B runs)
  static const bool off = getenv("FFMI_SKINNY_SPLIT") && atoi(getenv("FFMI_SKINNY_SPLIT")) == 0;
  if (off || !deferrable || epi || T > 64) return 1;
  const int ntiles = (N + 15) / 16;
  const int KT = K / 32;
  if (ntiles >= 128) {
    const auto evens = [](int wgs) { return (2 * wgs + 255) / 256 < 2 * ((wgs + 255) / 256); };
    if (KT < 32 || (ntiles >= 1024 && KT <= 32)) return 1;
    return evens(ntiles) && (ntiles < 512 || evens((ntiles + 1) / 2)) ? 2 : 1;
  }
  int S = 256 / ntiles;
  S = std::min(S, std::max(1, KT / 8));  // >= 1 k-step per wave of an 8-wave slice
  return std::max(1, std::min(S, 8));
}

// The fused residual/norm forms (FuseArgs; S == 1, T <= 16): the unfused
// path's tile and wave choices, one instantiation set per role.
template <int FZ>
static hipError_t dispatch_fused(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, int T, int N,
                                 int K, int KT, int epi, hipStream_t s, int xp, int yp, bool nt,
                                 int wpitch, const FuseArgs &fz) {
  constexpr int U = 8;
  const int ntiles = (N + 15) / 16;
  // FFMI_FZ_KW8 (A/B): 8 K-split waves instead of 4 for the consumer launches
  // -- 1: qkv, 2: qkv and gate/up
  static const int kw8 = getenv("FFMI_FZ_KW8") ? atoi(getenv("FFMI_FZ_KW8")) : 0;
  if (epi == FFMI_EPI_SILU_MUL) {
    if constexpr (FZ == 2) {
      if (kw8 >= 2)
        return run<1, 2, 8, U, 1, 2>(X, Wp, Y, nullptr, T, N, K, KT, 2 * ntiles, 1, s, xp, yp, nt,
                                     wpitch, fz);
      return run<1, 2, 4, U, 1, 2>(X, Wp, Y, nullptr, T, N, K, KT, 2 * ntiles, 1, s, xp, yp, nt,
                                   wpitch, fz);
    }
    return hipErrorInvalidValue;
  }
  if constexpr (FZ == 2)
    if (kw8 >= 1 && ntiles >= 512)
      return run<1, 1, 8, U, 0, FZ>(X, Wp, Y, nullptr, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch, fz);
  // FFMI_FZ_NT2=1: two tiles per workgroup (A/B)
  static const bool nt2 = getenv("FFMI_FZ_NT2") && atoi(getenv("FFMI_FZ_NT2")) != 0;
  if (nt2 && ntiles >= 512)
    return run<1, 2, 4, U, 0, FZ>(X, Wp, Y, nullptr, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch, fz);
  if (ntiles < 512 && KT >= 64 && !nt)
    return run<1, 1, 8, U, 0, FZ>(X, Wp, Y, nullptr, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch, fz);
  return run<1, 1, 4, U, 0, FZ>(X, Wp, Y, nullptr, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch, fz);
}

// E: the epilogue kind (1: paired tiles)
template <int E, int MT, int U>
static hipError_t dispatch_nt(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws,
                              int T, int N, int K, int KT, int S, hipStream_t s,
                              int xp, int yp, bool nt, int wpitch, const FuseArgs &fz) {
  int ntiles = (N + 15) / 16;
  if (!wpitch) wpitch = epi_paired<E> ? 2 * ntiles : ntiles;
  if constexpr (epi_paired<E>)
    return run<MT, 2, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, 2 * ntiles, 1, s, xp, yp, nt, wpitch, fz);
  else {
  // diagnostics: FFMI_SKINNY="NT,KW" forces the tile count and K-split waves
  // of every unsplit skinny launch (A/B runs, scripts/gemm_bench.py)
  static int fnt = -1, fkw = 0;
  if (fnt < 0) {
    fnt = 0;
    if (const char *e = getenv("FFMI_SKINNY")) (void)sscanf(e, "%d,%d", &fnt, &fkw);
  }
  if constexpr (E == 0) if (fnt > 0 && S == 1 && MT <= 2) {
    if (fnt == 1 && fkw == 4) return run<MT, 1, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 1 && fkw == 8) return run<MT, 1, 8, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 2 && fkw == 4) return run<MT, 2, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 2 && fkw == 8) return run<MT, 2, 8, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 4 && fkw == 4) return run<MT, 4, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 4 && fkw == 2) return run<MT, 4, 2, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
    if (fnt == 2 && fkw == 2) return run<MT, 2, 2, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, 1, s, xp, yp, nt, wpitch);
  }
  // wide, short-K layers (the SSM lm_head): one wave per 2 tiles over the
  // whole K (gemm_wave_kernel; FFMI_WAVE_GEMM=0 keeps the K-split form)
  static const bool wave_ok = !getenv("FFMI_WAVE_GEMM") || atoi(getenv("FFMI_WAVE_GEMM")) != 0;
  if (wave_ok && ntiles >= 1024 && KT <= 32 && S == 1) {
    const size_t wts = w_tile_stride(KT), wks = w_k_stride(wpitch);
    // two tiles per wave: SSM lm_head (32000 x 768) at T = 24 11.1 us (13.3
    // in the K-split form, 13.3 with one tile per wave and twice the waves),
    // T = 8 9.4 us (12.5)
    // (FFMI_WAVE_FORM=NT,WPG: tiles per wave and waves per workgroup, A/B)
    static int wnt = 2, wpg = 4;
    static bool wread = false;
    if (!wread) {
      wread = true;
      if (const char *e = getenv("FFMI_WAVE_FORM")) (void)sscanf(e, "%d,%d", &wnt, &wpg);
    }
#define FFMI_WAVE(NTV, WPGV, NL)                                                               \
  hipLaunchKernelGGL((gemm_wave_kernel<MT, NTV, 4, NL, WPGV, E>),                              \
                     dim3(((ntiles + NTV - 1) / NTV + WPGV - 1) / WPGV), dim3(WPGV * 64), 0, s, X, \
                     Wp, Y, ws, T, N, KT, ntiles, xp, yp, wts, wks, NoArgs())
    if constexpr (E >= 2) {
      if (nt) FFMI_WAVE(2, 4, true);
      else FFMI_WAVE(2, 4, false);
    } else if (wnt == 4 && wpg == 2) {
      if (nt) FFMI_WAVE(4, 2, true);
      else FFMI_WAVE(4, 2, false);
    } else if (wnt == 4 && wpg == 4) {
      if (nt) FFMI_WAVE(4, 4, true);
      else FFMI_WAVE(4, 4, false);
    } else if (wnt == 3 && wpg == 2) {
      if (nt) FFMI_WAVE(3, 2, true);
      else FFMI_WAVE(3, 2, false);
    } else if (wnt == 2 && wpg == 2) {
      if (nt) FFMI_WAVE(2, 2, true);
      else FFMI_WAVE(2, 2, false);
    } else {
      if (nt) FFMI_WAVE(2, 4, true);
      else FFMI_WAVE(2, 4, false);
    }
#undef FFMI_WAVE
    return hipGetLastError();
  }
  // wide layers (lm_head): two tiles per workgroup once there are >= 2 row
  // tiles (SSM lm_head at T = 24: 16.1 -> 12.3 us warm), or more than half of one
  // and tiles for three rounds of pairs (cold, 9 to 16 rows alike: 32000 x 4096
  // 48.8 -> 40.8 us, 24576 x 4096 34.3 -> 31.8, 50272 x 4096 71.0 -> 66.2, 128256 x
  // 4096 179 -> 169; at 16 rows 20480 x 4096 30.6 -> 31.3, 12288 x 4096 19.5 ->
  // 21.5).  Up to 8 rows a single tile is the faster for most widths (12288 to
  // 128256 x 4096 lose 4-13 %, 32000 gains 8)
  if (MT >= 2 ? ntiles >= 512 : T > 8 && ntiles >= 1536)
    return run<MT, 2, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, xp, yp, nt, wpitch);
  // 8-wave groups only where the accumulators fit 2 waves/SIMD (no spills)
  if (ntiles >= 512 || MT >= 8)
    return run<MT, 1, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, xp, yp, nt, wpitch);
  // ... and where each wave still gets a full batch of U k-steps (K = 768 of
  // the SSM: 4 waves x 6 k-steps beat 8 x 3, qkv T = 24: 5.7 -> 4.2 us).
  // Non-temporal weight loads (FFMI_W_STREAM) keep 4 waves at every row-tile
  // count (LLaMA-7B decode, cold, T = 1-16: o 7.6-8.8 -> 7.2-8.6 us, down
  // 17.0-24.8 -> 16.4-21.9 us over two runs of gemm_bench.py --wstream; T = 32
  // within noise), so a row's reduction order still depends on (N-tile, K,
  // policy) only, not on T: the threshold is a fixed 64 k-steps per slice
  // (8 waves x the largest batch U = 8), never U itself, which depends on T.
  if ((KT + S - 1) / S >= 64 && !nt)
    return run<MT, 1, 8, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, xp, yp, nt, wpitch);
  return run<MT, 1, 4, U, E>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, xp, yp, nt, wpitch);
  }
}

// ---------------------------------------------------------------------------
// M-split GEMM for 64 < T <= 192 (verify batches, small prompts; msplit_ahead).
//
// The skinny kernel above re-reads the whole activation block from L2 in
// every wave (K split over waves) and runs at 1 wave/SIMD at T ~ 168, which
// made it latency-bound (~0.7 TB/s).  Here the 4 waves of a workgroup split
// the ROWS (MTW m-tiles each, 64*MTW rows per block) and share one weight
// tile of NTW 16-column tiles per 32-deep k-step, staged through LDS with a
// register double buffer (load k+1 while the MFMAs of k run, one barrier per
// k-step).  Each wave loads only its own rows of X.  Small-N layers are
// split over K across workgroups (S slices, fp32 partials reduced in slice
// order by gemm_reduce_kernel), so every layer puts >= ~256 workgroups on
// the 256 CUs.  Reduction order per output element: MFMA chain over the
// slice's k-steps, then slices 0..S-1 -- fixed by (N, K, S), not by T.
// ---------------------------------------------------------------------------
// Epilogue of the M-split kernel.  Its MFMAs compute D = W_tile . X_tile^T,
// so a lane's accumulator holds FOUR CONSECUTIVE OUTPUT COLUMNS
// n = tile*16 + (lane>>4)*4 + r of one row m = m0 + i*16 + (lane&15): the
// fp16 output goes out as one 8-byte store and an fp32 partial as one 16-byte
// store per (i, j) (scalar 2-/4-byte stores in the C layout were the
// kernel's single largest cost).
template <int MTW, int NTW, int EPI>
__device__ __forceinline__ void mid_store(const f4 (&acc)[MTW][NTW], uint16_t *__restrict__ Y,
                                          float *__restrict__ Ypart, int T, int N, int NTILES,
                                          int S, int ks, int tile0, int m0, int lane, int yp,
                                          float lim) {
  const int mr = lane & 15, nq = (lane >> 4) * 4;
  if (S > 1 || epi_f32<EPI>) {
    const int NP = NTILES * 16;
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
      const int tile = tile0 + j;
      if (tile >= NTILES) continue;
#pragma unroll
      for (int i = 0; i < MTW; ++i) {
        const int m = m0 + i * 16 + mr;
        if (m < T)
          // (non-temporal stores here measured slower end to end: the
          // consumer then reads the slabs from memory instead of L2)
          *reinterpret_cast<f4 *>(Ypart + ((size_t)ks * T + m) * NP + tile * 16 + nq) = acc[i][j];
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < NTW; j += (epi_paired<EPI> ? 2 : 1)) {
    const int tile = tile0 + j;
    if (tile >= NTILES) continue;
    const int n = (epi_paired<EPI> ? (tile >> 1) : tile) * 16 + nq;
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < MTW; ++i) {
      const int m = m0 + i * 16 + mr;
      if (m >= T) continue;
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if constexpr (epi_paired<EPI>) o[r] = pair16<EPI>(acc[i][j][r], acc[i][j + 1][r], lim);
        else o[r] = out16<EPI>(acc[i][j][r]);
      uint16_t *dst = yp ? Y + act_packed_off(m, n, yp) : Y + (size_t)m * N + n;
      if (n + 4 <= N && (((uintptr_t)dst & 7) == 0)) {
        *reinterpret_cast<uint2 *>(dst) =
            make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) dst[r] = o[r];
      }
    }
  }
}

// Diagnostic stamps (FFMI_GEMM_STAMP=1 builds only): per wave
// {realtime start, after prologue, after k-loop, end, HW_ID, XCC_ID, core-clock
// counter (s_memtime) after prologue, after k-loop}; realtime is 100 MHz, so
// the k-loop's clock = d(memtime) / d(realtime) x 100 MHz.
static __device__ long long *g_gemm_stamps;
__device__ __forceinline__ long long rt_now() { return __builtin_amdgcn_s_memrealtime(); }

template <int MTW, int NTW, int PF, int EPI, bool STAMP = false, bool XP = false, bool ULD = false,
          bool NTL = false>
// (two workgroups per CU = 256 registers per wave: up to 24 accumulator tiles,
// MTW x NTW)
__global__ __launch_bounds__(256, NTW <= 8 && MTW * NTW <= 24 ? 2 : 1) void gemm_mid_kernel(
    const uint16_t *__restrict__ X, const uint16_t *__restrict__ Wp,
    uint16_t *__restrict__ Y, float *__restrict__ Ypart, int T, int N, int K, int KT,
    int NTILES, int S, int yp, size_t wts, size_t wks, float lim) {
  long long st0 = 0, st1 = 0, st2 = 0, ck1 = 0, ck2 = 0;
  if (STAMP) st0 = rt_now();
  static_assert(NTW % 2 == 0, "gate/up tiles come in pairs");
  static_assert(PF >= 2, "ring depth");
  // weight tiles j = wave + 4p are loaded by wave (j % 4); with NTW % 4 != 0
  // the last round is loaded by the first NTW % 4 waves only
  constexpr int PPT = (NTW + 3) / 4;
  __shared__ __attribute__((aligned(16))) h8 sB[2][NTW][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int tile0 = blockIdx.x * NTW;
  const int ks = blockIdx.y;
  const int m0 = blockIdx.z * (4 * MTW * 16) + wave * MTW * 16;
  const int per = (KT + S - 1) / S;
  const int kb = min(KT, ks * per);
  const int ke = min(KT, kb + per);

  const uint16_t *bsrc[PPT];
  int bj[PPT];
#pragma unroll
  for (int p = 0; p < PPT; ++p) {
    bj[p] = wave + 4 * p;
    // ULD: waves past the last tile re-load the block's last tile (an L2 hit
    // beside the wave that owns it) so that EVERY wave issues PPT weight loads
    // per k-step: loads behind a wave-dependent branch are invisible to the
    // compiler's vmcnt counting, which then waits for ~2 ring slots, not PF-1
    const int t = min(tile0 + (ULD ? min(bj[p], NTW - 1) : bj[p]), NTILES - 1);
    bsrc[p] = Wp + (size_t)t * wts + lane * 8;
  }
  // X row-major [T][K] (16 rows x 64 B per fragment load), or XP: packed
  // activation tiles [T/16][KT][64 lanes][8] (one contiguous 1 KiB per load)
  constexpr int XS = XP ? 512 : 32;  // halves per k-step
  const uint16_t *xrow[MTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i) {
    if (XP) {
      const int mt = min((m0 + i * 16) >> 4, (T - 1) >> 4);
      xrow[i] = X + ((size_t)mt * KT * 64 + lane) * 8;
    } else {
      const int r = min(m0 + i * 16 + (lane & 15), T - 1);
      xrow[i] = X + (size_t)r * K + 8 * (lane >> 4);
    }
  }
  f4 acc[MTW][NTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};

  // Software pipeline, one barrier per 32-deep k-step.  A PF-deep register
  // ring holds BOTH operands of k-steps k..k+PF-1: slot q = (X(k), B(k)).
  // Loads retire in issue order (vmcnt), so X must be issued as early as the
  // weights: X(k) is consumed PF steps after issue, B(k+1) goes to the LDS
  // tile PF-1 steps after issue, and no consumer waits on a young load.
  auto kloop = [&](auto NVc) {
    constexpr int NV = decltype(NVc)::value;
    h8 bq[PF][PPT];
    h8 xq[PF][MTW];
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      const int kq = min(kb + q, ke - 1);
#pragma unroll
      for (int i = 0; i < NV; ++i) xq[q][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)kq * XS);
#pragma unroll
      for (int p = 0; p < PPT; ++p)
        if (ULD || NTW % 4 == 0 || bj[p] < NTW) bq[q][p] = ld_weight<NTL>(bsrc[p] + (size_t)kq * wks);
    }
#pragma unroll
    for (int p = 0; p < PPT; ++p)
      if (NTW % 4 == 0 || bj[p] < NTW) sB[0][bj[p]][lane] = bq[0][p];
    __syncthreads();
    if (STAMP) st1 = rt_now(), ck1 = __builtin_amdgcn_s_memtime();
    // one k-step on ring slot Q; MFMAs read the slot in place, then it is
    // refilled (a copy would rotate the ring through fresh registers and
    // force vmcnt drains at the loop back-edge)
    int cur = 0;
    auto step = [&](auto Qc, int kt) {
      constexpr int Q = decltype(Qc)::value;
      h8 b[NTW];
#pragma unroll
      for (int j = 0; j < NTW; ++j) b[j] = sB[cur][j][lane];
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j)  // D = W . X^T (see mid_store)
          acc[i][j] = mma16<EPI>(b[j], xq[Q][i], acc[i][j]);
      const int kw = min(kt + PF, ke - 1);
#pragma unroll
      for (int i = 0; i < NV; ++i) xq[Q][i] = *reinterpret_cast<const h8 *>(xrow[i] + (size_t)kw * XS);
#pragma unroll
      for (int p = 0; p < PPT; ++p)
        if (ULD || NTW % 4 == 0 || bj[p] < NTW) bq[Q][p] = ld_weight<NTL>(bsrc[p] + (size_t)kw * wks);
      // B(kt+1) lives in ring slot (Q+1) % PF
#pragma unroll
      for (int p = 0; p < PPT; ++p)
        if (NTW % 4 == 0 || bj[p] < NTW) sB[cur ^ 1][bj[p]][lane] = bq[(Q + 1) % PF][p];
      __syncthreads();
      cur ^= 1;
    };
    int kt0 = kb;
    for (; kt0 + PF <= ke; kt0 += PF)  // steady state: whole ring turns
      static_for<PF>([&](auto Qc) { step(Qc, kt0 + decltype(Qc)::value); });
    static_for<PF - 1>([&](auto Qc) {  // tail: < PF steps, slots 0..
      if (kt0 + decltype(Qc)::value < ke) step(Qc, kt0 + decltype(Qc)::value);
    });
  };
  if (kb < ke) kloop(std::integral_constant<int, MTW>{});
  if (STAMP) st2 = rt_now(), ck2 = __builtin_amdgcn_s_memtime();

  mid_store<MTW, NTW, EPI>(acc, Y, Ypart, T, N, NTILES, S, ks, tile0, m0, lane, yp, lim);
  if (STAMP) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const long long st3 = rt_now();
    unsigned hwid, xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hwid));
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    if (lane == 0 && g_gemm_stamps) {
      const long b = blockIdx.x + (long)gridDim.x * (blockIdx.y + (long)gridDim.y * blockIdx.z);
      long long *d = g_gemm_stamps + (b * 4 + wave) * 8;
      d[0] = st0; d[1] = st1; d[2] = st2; d[3] = st3; d[4] = hwid; d[5] = xcc;
      d[6] = ck1; d[7] = ck2;
    }
  }
}

// Tile form of T > 192 (tile_plan, msplit_ahead), and with twelve waves of 65 .. 192 rows
// (takes_six): one workgroup per output tile of
// WR x MI row tiles by WC x NJ weight tiles, its WR x WC waves MI x NJ MFMA
// accumulators each.  Every operand fragment (16 x 32, 1 KiB) lands in LDS in
// the MFMA's order with ONE global_load_lds_dwordx4 wave-instruction
// (lane-linear: no swizzle, conflict-free ds_read_b128 reads) in a ring of NB
// one-k-step stages; weights and packed activations lie in that order
// (weights.hip, pack_act_kernel), of row-major ones each lane fetches its own
// 16 bytes.
//
// What bounds it: the matrix pipe, once the loop keeps it fed.  A CU takes in
// 120-148 GB/s from its L2 (256 x 256 tiles ask for 55), so bytes are not the
// limit; a k-step that reads its fragments after the barrier and multiplies
// them afterwards is (0.77 us per k-step of 256 x 256 against 0.43 of MFMA
// issue).  So:
//  * the fragments of step k + 1 are read while step k is multiplied, each
//    row's into the registers that its MFMAs have just used and the weight
//    fragments into a second set, with NB - 2 later stages in flight across
//    the barrier (a counted s_waitcnt vmcnt, never 0 in the steady state, and
//    a raw s_barrier: __syncthreads would drain the DMAs).  Waves of three rows and four
//    weight tiles or more (kTwoX) read the rows into a second set too, and all of it
//    ahead of the last row's MFMAs, so that no read is waited for at the step's end;
//  * the loop body has no branches (a step without a next one is a separate
//    instantiation; waves past the last fragment load it again, or see
//    kExactCopies), and
//    sched_barrier pins MFMA group / LDS read / DMA in turn: left alone the
//    compiler collects the reads behind the MFMAs and waits for them;
//  * a wave's MFMA groups run at raised priority, so that of the two waves of
//    a SIMD one multiplies while the other issues loads.
// 256 x 256: 0.77 -> 0.60 -> 0.56 us per k-step (pipelining, priority).
// T = 1024, cold weights, before (256 x 256 tiles unpipelined, M-split where
// those did not fill the chip) and now: N 12288 x K 4096 111-117 -> 91 us
// (1.13 PFLOP/s), gate/up 2 x 11008 222 -> 163, K 11008 x N 4096 108 -> 93,
// N 4096 x K 4096 48 -> 38, N 32000 256-269 -> 224-228.
// The k order of every accumulator is the M-split kernel's (k-steps in
// sequence, one MFMA each), so outputs are bit-identical to gemm_mid_kernel at
// equal splits of K.  Blocks are remapped so the row blocks of a weight tile
// and slice share an XCD (bijective remap): its weights come from HBM once per
// XCD L2.
// NTL (FFMI_W_STREAM, one row block: each weight is read once): non-temporal weight
// copies.  T = 216: K 11008 x N 4096 35.4 us either way, 12288 x 4096 39.2 and 39.1; with
// two row blocks the second one's reads miss (4096 x 4096 21.3 -> 25.3, gate/up 55.3
// -> 63.6), which therefore go without the hint.
// A stage whose fragments the waves do not share evenly: the last waves copy one less
// (an instance of the loop per count, and with NTL per kind; each waits for its own
// copies).  Twelve waves only, of which 6 and 10 would copy for nothing; the forms of eight gain nothing
// from it (400 products of 200 .. 1024 rows: 0.2% slower to 0.3% faster a form).
template <int MI, int NJ, int WR, int WC>
static constexpr bool kExactCopies = WR * WC > 8 && (MI * WR + NJ * WC) % (WR * WC) != 0;
// Two sets of row fragments.  One set / two, us, cold weights, both in turn three times.  192 x 128: 11264 x
// 2048 gate and up at 280 rows 31.9 / 30.6, 6144 x 2048 at 700 34.6 / 33.0.  256 x 128: 4096 x 11008 at 1024
// 110.5 / 109.3 (two slices), at 400 59.5 / 58.4 (four), 8192 x 2048 at 1024 44.3 / 43.2.  256 x 192: 22016 x 4096 at
// 1024 183 / 180, at 512 93.2 / 92.2, 11264 x 2048 at 1024 57.1 / 55.5, 12288 x 4096 at 700 86.9 / 85.4.  192 x 256:
// 22016 x 4096 at 280 81.7 / 81.0, 4096 x 11008 at 700 85 / 85.  256 x 256: 27648 x 5120 at 1024 264 / 263,
// 5120 x 13824 at 1024 160 / 155 (three slices).  One block of rows: 32000 x 4096 at 256 rows 77 - 80 / 79 - 81, weights
// streamed 82 - 91 / 72 - 76.  Two rows a wave gain nothing (4096 x 4096 in 128 x 128 40.3 / 40.9) or
// lose (6144 x 2048 in 128 x 192 31.9 / 32.6), as twelve waves do (22016 x 4096 at 168 rows 52.5 / 53.6).
template <int MI, int NJ, int WR, int WC>
static constexpr bool kTwoX = MI >= 3 && NJ >= 4 && WR * WC <= 8;
template <int EPI, int MI, int NJ, int WR, int WC, int NB, bool NTL>
__global__ __launch_bounds__(WR * WC * 64, 1) void gemm_tile_kernel(
    const uint16_t *__restrict__ X, const uint16_t *__restrict__ Wp, uint16_t *__restrict__ Y,
    float *__restrict__ Yf, int T, int N, int KT, int NTILES, int nbm, int S, int xp, int yp,
    size_t wts, size_t wks, float lim) {
  constexpr int NW = WR * WC, FX = MI * WR, F = FX + NJ * WC;  // waves; fragments of a stage
  constexpr int PMAX = (F + NW - 1) / NW;                      // DMAs per wave and stage
  static_assert(NB >= 3 && (NB - 1) * PMAX < 64, "stages in flight");
  static_assert(!NTL || FX % NW == 0 || (kExactCopies<MI, NJ, WR, WC> && F % NW <= FX % NW),
                "a wave's copy is of X or of weights, known to the compiler");
  __shared__ __attribute__((aligned(1024))) h8 lds[NB][F][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nwg = gridDim.x, b = blockIdx.x;
  const int xcd = b & 7, q = nwg >> 3, r = nwg & 7;
  const int L = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (b >> 3);
  const int bm = L % nbm, ks = L / nbm % S, bn = L / (nbm * S);
  // this slice's k-steps: [kb, kb + n), n >= 1 (tile_plan)
  const int per = (KT + S - 1) / S, kb = ks * per, n = min(KT, kb + per) - kb;
  const int wm = wave / WC, wn = wave % WC;
  f4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  auto loop = [&](auto PWc, auto PXc) __attribute__((always_inline)) {
    constexpr int PW = decltype(PWc)::value, PX = decltype(PXc)::value;
    // this wave's fragments f = wave + NW p of a stage: X row tile f (< FX) or
    // weight tile f - FX (the last rows / tile again past the end); NTL: the first PX
    // of X, the others of weights
    const uint16_t *src[PW];
    size_t step[PW];
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      const int f = min(wave + NW * p, F - 1);
      if (f >= FX) {
        src[p] = Wp + (size_t)min(bn * (F - FX) + f - FX, NTILES - 1) * wts + (size_t)kb * wks + lane * 8;
        step[p] = wks;
      } else if (xp) {
        src[p] = X + ((size_t)min(bm * FX + f, (T - 1) >> 4) * KT + kb) * 512 + lane * 8;
        step[p] = 512;
      } else {
        const int row = min((bm * FX + f) * 16 + (lane & 15), T - 1);
        src[p] = X + ((size_t)row * KT + kb) * 32 + 8 * (lane >> 4);
        step[p] = 32;
      }
    }
    auto issue = [&](int kt, int slot, int p) {
      const auto from = (const __attribute__((address_space(1))) void *)(src[p] + (size_t)kt * step[p]);
      const auto to = (__attribute__((address_space(3))) void *)(&lds[slot][min(wave + NW * p, F - 1)][0]);
      // (cache policy 2: non-temporal)
      if (NTL && p >= PX) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2);
      else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    };
    // (fewer steps than stages: the last step again, into slots nobody reads)
#pragma unroll
    for (int kt = 0; kt < NB; ++kt) {
#pragma unroll
      for (int p = 0; p < PW; ++p) issue(min(kt, n - 1), kt, p);
    }
    constexpr bool TWO = kTwoX<MI, NJ, WR, WC>;
    h8 xa[MI], x2[TWO ? MI : 1], wa[NJ], wb[NJ];
    auto &xb = [&]() -> h8(&)[MI] {
      if constexpr (TWO) return x2;
      else return xa;
    }();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 1) * PW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NJ; ++j) wa[j] = lds[0][FX + wn * NJ + j][lane];
#pragma unroll
    for (int i = 0; i < MI; ++i) xa[i] = lds[0][wm * MI + i][lane];
    int slot = 0;
    // Step kt on xc / wc, with step kt + 1's fragments read into xx / wx.  The
    // wait leaves the NB - 2 stages after kt + 1 in flight and retires this
    // wave's own reads of stage kt (issued a step ago); behind the barrier stage
    // kt + 1 is there for every wave and stage kt's slot is free for kt + NB.
    // MORE: step kt + NB exists.  (The last step reads a stale slot unused.)
    auto kstep = [&](auto MOREc, h8(&xc)[MI], h8(&wc)[NJ], h8(&xx)[MI], h8(&wx)[NJ], int kt) {
      constexpr bool MORE = decltype(MOREc)::value;
      constexpr int VM = MORE ? (NB - 2) * PW : 0;
      constexpr int R = MI + NJ, G = MI > 1 ? MI - 1 : 1;  // reads; the rows they go with (TWO)
      const int nslot = slot + 1 == NB ? 0 : slot + 1;
      // s_waitcnt vmcnt(VM) lgkmcnt(0)
      __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if constexpr (TWO) {
#pragma unroll
          for (int f = min(i, G) * R / G; f < min(i + 1, G) * R / G; ++f)
            if (f < NJ) wx[f] = lds[nslot][FX + wn * NJ + f][lane];
            else xx[f - NJ] = lds[nslot][wm * MI + f - NJ][lane];
        }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < NJ; ++j)  // D = W . X^T (see mid_store)
          acc[i][j] = mma16<EPI>(wc[j], xc[i], acc[i][j]);
        if constexpr (!TWO) {
          xx[i] = lds[nslot][wm * MI + i][lane];
#pragma unroll
          for (int j = i * NJ / MI; j < (i + 1) * NJ / MI; ++j) wx[j] = lds[nslot][FX + wn * NJ + j][lane];
        }
        if constexpr (MORE) {
#pragma unroll
          for (int p = i * PW / MI; p < (i + 1) * PW / MI; ++p) issue(kt + NB, slot, p);
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = nslot;
    };
    const auto yes = std::integral_constant<bool, true>{};
    const auto no = std::integral_constant<bool, false>{};
    int kt = 0;
    for (; kt + 2 + NB <= n; kt += 2) {
      kstep(yes, xa, wa, xb, wb, kt);
      kstep(yes, xb, wb, xa, wa, kt + 1);
    }
    if (kt + 1 + NB <= n) {
      kstep(yes, xa, wa, xb, wb, kt++);
#pragma unroll
      for (int j = 0; j < NJ; ++j) wa[j] = wb[j];
#pragma unroll
      for (int i = 0; i < MI; ++i) xa[i] = xb[i];
    }
#pragma unroll 1
    for (; kt < n; ++kt) {
      kstep(no, xa, wa, xb, wb, kt);
#pragma unroll
      for (int j = 0; j < NJ; ++j) wa[j] = wb[j];
#pragma unroll
      for (int i = 0; i < MI; ++i) xa[i] = xb[i];
    }
  };
  constexpr std::integral_constant<int, PMAX> most{};
  constexpr std::integral_constant<int, FX / NW> xs{};
  if constexpr (kExactCopies<MI, NJ, WR, WC>) {
    constexpr std::integral_constant<int, PMAX - 1> less{};
    if constexpr (!NTL || FX % NW == 0) {
      if (wave < F % NW) loop(most, xs);
      else loop(less, xs);
    } else {  // (a third instance: the last waves copy weights only)
      constexpr std::integral_constant<int, FX / NW + 1> more{};
      if (wave < F % NW) loop(most, more);
      else if (wave < FX % NW) loop(less, more);
      else loop(less, xs);
    }
  } else {
    loop(most, xs);
  }
  mid_store<MI, NJ, EPI>(acc, Y, Yf, T, N, NTILES, S, ks, bn * (F - FX) + wn * NJ,
                         (bm * FX + wm * MI) * 16, lane, yp, lim);
}

static inline long long *stamp_buf() {
  static long long *buf = nullptr;
  if (!buf) {
    if (hipMalloc(&buf, (size_t)8 << 20) != hipSuccess) return nullptr;
    (void)hipMemcpyToSymbol(HIP_SYMBOL(g_gemm_stamps), &buf, sizeof(buf));
  }
  return buf;
}
static long g_stamp_entries = 0;


// Sum the S fp32 partial slabs in slice order, then the epilogue; one thread
// per 4 consecutive output columns (16-B slab loads, 8-B fp16 store).
template <int EPI, int MAXS>
__global__ void gemm_reduce_kernel(const float *__restrict__ Ypart, uint16_t *__restrict__ Y,
                                   int T, int N, int NTILES, int S, int yp, float lim) {
  const int NP = NTILES * 16;
  const int nq = (N + 3) / 4;
  const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (idx >= (long)T * nq) return;
  const int m = (int)(idx / nq), n = (int)(idx % nq) * 4;
  const size_t slab = (size_t)T * NP;
  f4 acc, up;
  // all MAXS >= S slab loads go out before the first add (one memory round
  // trip, not S); indices past S re-read the last slab and are not added
  f4 pa[MAXS], pu[MAXS];
  const float *src = !epi_paired<EPI> ? Ypart + (size_t)m * NP + n
                              : Ypart + (size_t)m * NP + (n >> 4) * 32 + (n & 15);
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
    const float *q = src + (size_t)min(s, S - 1) * slab;
    pa[s] = *reinterpret_cast<const f4 *>(q);
    if (epi_paired<EPI>) pu[s] = *reinterpret_cast<const f4 *>(q + 16);
  }
  acc = pa[0];
  if (epi_paired<EPI>) up = pu[0];
#pragma unroll
  for (int s = 1; s < MAXS; ++s)
    if (s < S) {
      acc += pa[s];
      if (epi_paired<EPI>) up += pu[s];
    }
  uint16_t o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    o[r] = epi_paired<EPI> ? pair16<EPI>(acc[r], up[r], lim) : out16<EPI>(acc[r]);
  uint16_t *dst = yp ? Y + act_packed_off(m, n, yp) : Y + (size_t)m * N + n;
  if (n + 4 <= N && (((uintptr_t)dst & 7) == 0)) {
    *reinterpret_cast<uint2 *>(dst) =
        make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
  } else {
    for (int r = 0; r < 4; ++r)
      if (n + r < N) dst[r] = o[r];
  }
}

// Launch plan of the M-split kernel: weight tiles per workgroup (NTW) and
// split-K factor (S).  Each workgroup is bound by its CU's load path (per-wave
// timeline, scripts/diag_stamps.py: a k-step moves NTW KiB of weights + 4*MTW
// KiB of activations at ~50 GB/s per CU; two workgroups on one CU each run at
// half speed), so the plan keeps the grid within one wave of 256 workgroups,
// prefers wide tiles (fewer activation bytes per weight byte) and charges the
// split-K reduce pass.  Times in us; only the ranking matters.
struct MidPlan {
  int MTW, NTW, S, mblocks, nblk;
};
static MidPlan mid_plan(int T, int N, int K, int epi, bool deferred = false) {
  MidPlan p;
  const int mtiles = (T + 15) / 16;
  p.MTW = mtiles <= 8 ? 2 : 3;  // row tiles per wave: 4 waves x MTW tiles cover one row block
  p.mblocks = (mtiles + 4 * p.MTW - 1) / (4 * p.MTW);
  const int KT = K / 32;
  const int ntiles = (N + 15) / 16 * (epi ? 2 : 1);
  double best = 1e30;
  p.NTW = 8, p.S = 1;
  // measured k-step times (us) at MTW = 3, packed activations (diag_stamps.py)
  // (2 and 4: narrow per-rank shards of tensor parallelism, e.g. LLaMA-7B
  // o_proj at TP = 8 is 256 tiles x K = 512 -- 43 workgroups at NTW = 6)
  static const int ntw_opts[6] = {2, 4, 6, 8, 12, 16};
  static const double base[6] = {0.27, 0.30, 0.36, 0.40, 0.65, 0.90};
  static const int nopt = getenv("FFMI_MID_NARROW") && atoi(getenv("FFMI_MID_NARROW")) == 0 ? 4 : 6;
  for (int o = 6 - nopt; o < 6; ++o) {
    const int ntw = ntw_opts[o];
    const int nblk = (ntiles + ntw - 1) / ntw;
    for (int S = 1; S <= 8 && S <= KT; ++S) {
      const long wgs = (long)nblk * S * p.mblocks;
      const double rounds = (double)((wgs + 255) / 256);
      const double steps = (double)((KT + S - 1) / S);
      const double tstep = base[o] * (ntw + 4.0 * p.MTW) / (ntw + 12.0);
      double t = rounds * (steps * tstep + 4.0);
      const double slab_mb = (double)S * T * ntiles * 16 * 4 / 1e6;
      // slabs cost their write here and their read in the consumer; a
      // deferred read (norm / attention prologue) is no cheaper than the
      // reduce pass's: /6 had picked 8 slabs for LLaMA-7B o_proj at T = 168,
      // 4 tiles x 4 slabs ran 0.6 % faster end to end (3 of 3 A/B pairs)
      // (the SiLU reduce pass re-reads the gate AND up slabs: at the verify
      // size, 9-12 row tiles in one block, a forced-plan sweep of the TP = 8
      // gate/up shard put 4 tiles x 4-5 slabs at 18.4-18.9 us against 21.7
      // for the 6 x 8 the /3 charge picked, profiles/r06_tp8_gateup_plans.log;
      // the TP 1 / 2 / 4 and 65B TP 8 picks are unchanged by /2)
      const double slab_rate = epi && p.MTW == 3 && p.mblocks == 1 ? 2.0 : 3.0;
      if (S > 1) t += deferred ? slab_mb / 3.0 : 3.0 + slab_mb / slab_rate;
      if (t < best - 1e-9) best = t, p.NTW = ntw, p.S = S;
    }
  }
  // >= 4 row blocks (FFMI_TILE_GEMM=0 only): the k-step model above is
  // calibrated at T = 168
  if (p.mblocks >= 4 && !(deferred && ntiles <= 8)) {
    p.NTW = 8;
    p.S = K >= 8192 && KT >= 2 ? 2 : 1;
  }
  // diagnostics: FFMI_GEMM_PLAN="NTW,S" forces the tile width and split of
  // every M-split launch; "N:K:NTW,S;..." only of the listed shapes
  static const char *force = getenv("FFMI_GEMM_PLAN");
  if (force) {
    const char *q = force;
    while (q && *q) {
      int a = 0, b = 0, c = 0, d = 0, ntw = 0, S = 0;
      const int n = sscanf(q, "%d:%d:%d,%d", &a, &b, &c, &d);
      if (n == 4 && a == N && b == K) ntw = c, S = d;
      else if (n != 4 && sscanf(q, "%d,%d", &a, &b) == 2) ntw = a, S = b;
      if ((ntw == 2 || ntw == 4 || ntw == 6 || ntw == 8 || ntw == 12 || ntw == 16) && S >= 1 &&
          S <= std::min(KT, 8)) {
        p.NTW = ntw, p.S = S;
        break;
      }
      q = strchr(q, ';');
      if (q) ++q;
    }
  }
  p.nblk = (ntiles + p.NTW - 1) / p.NTW;
  return p;
}

// The tile kernel's forms (MI, NJ, WR, WC, NB) and what one costs in us, with
// `rounds` of 256 workgroups and the k-steps of a slice:
//   c0 + c1 (rounds - 1) + steps (a0 + a1 (rounds - 1) + b workgroups / 256)
//   + w per MB written + 0.22 per MB of slabs read by who sums them
// fitted (non-negative least squares on relative errors, 4-8% rms) to 5500
// timings of every form and split at T = 72 .. 1024 on N x K of 2048 x 2048,
// 6144 x 2048, 2 x 5632 x 2048, 2048 x 5632 and twice as wide, and 32000 x
// 4096, cold weights.  The form that the estimate picks was 1.2% off the
// fastest of all on average.
struct TileForm {
  int MI, NJ, WR, WC, NB;
  double c0, c1, a0, a1, b, w;
};
static constexpr TileForm kTileForms[] = {
    {2, 2, 4, 2, 5, 3.305, 0.000, 0.136, 0.129, 0.046, 0.172},
    {3, 2, 2, 4, 8, 3.903, 1.631, 0.153, 0.161, 0.076, 0.158},
    {2, 4, 4, 2, 4, 3.823, 0.453, 0.193, 0.144, 0.087, 0.185},
    {2, 6, 4, 2, 7, 5.698, 2.602, 0.255, 0.259, 0.126, 0.156},
    {3, 4, 4, 2, 7, 4.482, 1.550, 0.263, 0.275, 0.119, 0.196},
    {4, 4, 2, 4, 6, 6.137, 3.600, 0.306, 0.309, 0.159, 0.131},
    {4, 4, 4, 2, 6, 4.528, 1.493, 0.308, 0.322, 0.135, 0.206},
    {4, 6, 4, 2, 5, 6.085, 2.386, 0.423, 0.444, 0.182, 0.183},
    {6, 4, 2, 4, 5, 6.780, 4.624, 0.413, 0.423, 0.201, 0.162},
    {8, 4, 2, 4, 4, 7.088, 4.426, 0.505, 0.551, 0.236, 0.168}};
static constexpr int kNumTileForms = sizeof(kTileForms) / sizeof(kTileForms[0]);
struct TilePlan {
  int form, S, nbm, nbn;
  bool msplit[2];  // [packed activations]: the M-split kernel is the faster one (msplit_ahead)
};
// Where the M-split kernel stays ahead of the tile forms (us).
//  * Up to 192 rows, one row block whose non-temporal weight stream is the time (in
//    the model, at T = 168, o_proj and down with the norms that read their slabs 55.7
//    against 57.2, N 32000 x K 4096 58 against 65, 12288 x 4096 32 against 36; at
//    T = 82 K 9600 x N 4096 20.0 against 23.7).
//  * Two blocks of up to 192 rows of a large unpaired weight (12288 x 4096 at T = 384
//    46.3 against 51.6, 4096 x 11008 44.9 against 47.5; but gate/up 90.6 against 78.8).
//  * Two such blocks of a small product of packed activations: narrow waves, all in
//    one round, up to 44 k-steps a slice and as many slices as the tiles take (so that
//    row-major and packed activations give the same bits).  The tile kernel fills its
//    ring of stages first, which costs it about 0.5 us and is not won back in so few
//    steps.  At T = 257 and 384: 2304 x 768 7.1 and 7.2 against 7.6, 2048 x 512 5.8 and 6.0
//    against 6.3 and 6.4, 8192 x 1024 10.8 and 10.3 against 11.2, 512 x 4096 10.2 and 11.3 against
//    10.8 and 11.8; but 768 x 768, split by one kernel only, 8.4 and 8.5 against 7.2, and 6144 x 2048,
//    longer slices, 20.1 and 20.1 against 20.0 and 20.2.  Row-major operands cost the M-split
//    kernel more than that (2304 x 768 12.6 against 10.6, 8192 x 1024 16.8 against 13.8).
static bool msplit_ahead(int mtiles, int ntiles, int N, int K, bool paired, bool xp, bool deferred, const TilePlan &t) {
  if (mtiles <= 12) return true;
  if (mtiles <= 16 || mtiles > 24) return false;
  if ((long)ntiles * 16 * K >= 1L << 25) return !paired && ntiles <= 1024;
  if (!xp) return false;
  const MidPlan m = mid_plan(mtiles * 16, N, K, paired, deferred && !paired);
  const int steps = (K / 32 + m.S - 1) / m.S;
  return m.NTW <= 4 && steps <= 44 && (long)m.nblk * m.S * m.mblocks <= 256 && m.S == t.S;
}
// f32: the output is slabs in any case; deferred: the consumer sums the slabs
// (else a reduce pass).  Depends on T by its row tiles only, as workspaces are
// sized.  The search takes about a microsecond; a thread keeps what it found,
// by sizes alone.
static TilePlan tile_plan(int T, int N, int K, bool paired, bool f32, bool deferred) {
  const int mtiles = (T + 15) / 16, ntiles = (N + 15) / 16 * (paired ? 2 : 1), KT = K / 32;
  struct Found {
    int mtiles = 0, ntiles = 0, KT = 0, flags = 0;
    TilePlan plan[2];  // [deferred]
  };
  static thread_local Found found[1024];
  const int flags = (paired ? 1 : 0) | (f32 ? 2 : 0);
  Found &at = found[(((mtiles * 4u + flags) * 0x9E3779B1u) ^ (ntiles * 0x85EBCA6Bu) ^ (KT * 0xC2B2AE35u)) >> 22];
  if (at.mtiles == mtiles && at.ntiles == ntiles && at.KT == KT && at.flags == flags) return at.plan[deferred];
  const double mb = mtiles * 16e-6 * ntiles * 16;  // million sums
  TilePlan best[2] = {};
  double least[2] = {1e30, 1e30};
  for (int f = 0; f < kNumTileForms; ++f) {
    const TileForm &F = kTileForms[f];
    const int nbm = (mtiles + F.MI * F.WR - 1) / (F.MI * F.WR), nbn = (ntiles + F.NJ * F.WC - 1) / (F.NJ * F.WC);
    for (int S = 1; S <= 8 && S <= KT; ++S) {
      const int steps = (KT + S - 1) / S;
      const long wgs = (long)nbm * nbn * S, rounds = (wgs + 255) / 256;
      // (no slice without k-steps, no split of what fills the chip twice)
      if (S > 1 && wgs > 640) break;
      if (S > 1 && (S - 1) * steps >= KT) continue;
      double t = F.c0 + F.c1 * (rounds - 1) + steps * (F.a0 + F.a1 * (rounds - 1) + F.b * wgs / 256.0);
      t += F.w * mb * (S > 1 || f32 ? 4.0 * S : paired ? 1.0 : 2.0);
      if (S > 1) t += 4.0 * S * mb / 4.5;
      for (int d = 0; d < 2; ++d)
        if (t + (S > 1 && !d ? 3.0 : 0.0) < least[d])
          least[d] = t + (S > 1 && !d ? 3.0 : 0.0), best[d] = TilePlan{f, S, nbm, nbn, {}};
    }
  }
  for (int d = 0; d < 2; ++d)
    for (int x = 0; x < 2; ++x) best[d].msplit[x] = msplit_ahead(mtiles, ntiles, N, K, paired, x, d, best[d]);
  at = Found{mtiles, ntiles, KT, flags, {best[0], best[1]}};
  return best[deferred];
}
// FFMI_TILE_GEMM: 0 never, 2 whatever the size (A/B runs and tests; read per call)
static int tile_mode() {
  const char *e = getenv("FFMI_TILE_GEMM");
  return e ? atoi(e) : 1;
}
static bool use_tiles(int T, int N, int K, bool paired, bool xp, bool f32, bool deferred) {
  const int mode = tile_mode();
  if (mode != 1) return mode == 2;
  return T > 192 && !tile_plan(T, N, K, paired, f32, deferred).msplit[xp];
}

// Unsplit products of 65 .. 192 rows of which the M-split plan gives a workgroup six weight
// tiles (96 columns): its waves then hold 2 or 3 x 6 accumulators and each copies six KiB of
// weights and its own rows a step, one stage ahead.  Twelve waves, 2 or 3 x 2
// accumulators each, keep 3 or 4 stages in flight and share every copy.  Cold streamed
// weights behind a norm, M-split / this at T = 72, 128, 168, 192 (us), on the better and on the
// worse of two machines: gate/up 2 x 11008 x 4096 40.2 / 39.0, 45.6 / 41.0, 51.3 / 47.5, 52.4 / 47.9
// and 42.1 / 40.5, 45.9 / 43.8, 52.1 / 50.3, 53.7 / 50.0; 20480 x 4096 40.5 / 35.2, 45.5 / 41.4, 51.0 / 46.2,
// 52.0 / 47.0 and 41.9 / 36.7, 45.8 / 42.4, 51.4 / 47.7, 52.9 / 48.2; 2 x 9216 x 1024 15.0 / 12.3, 15.1 / 13.4,
// 17.7 / 15.5, 17.9 / 15.7 and 15.1 / 13.1, 15.2 / 13.9, 18.1 / 16.3, 18.6 / 16.4; 24576 x 8192 at 168 97.5 / 91.3
// and 99.6 / 96.5.  Without the hint of a stream 0 to 10% less, 0.95 at worst.
// In K slices it depends on the machine, so those stay with the M-split kernel:
// 12288 x 4096 in two at T = 168 30.6 / 29.1 on one, 31.1 / 32.9 on the other (in the model 31.5 / 30.0
// and 32.0 / 33.7; T = 72 23.8 / 22.5 and 24.9 / 28.4), 6144 x 4096 in four 19.6 / 19.8 and 19.6 / 23.3, 2 x 3072 x 4096 in
// four 18.8 / 19.2 and 19.7 / 22.9.
// Where the plan has other widths the M-split kernel stays ahead of every form tried
// (32000 x 4096 at T = 168, 128 columns, 62.9 against 62.2 .. 91).
// Packed activations; not where the M-split kernel is to write its timeline
// (FFMI_GEMM_STAMP), nor without the tile kernel (FFMI_TILE_GEMM=0).
static bool takes_six(int T, int K, int NTW, int S, bool packed) {
  static const bool stamp = getenv("FFMI_GEMM_STAMP") != nullptr;
  return packed && !stamp && K % 32 == 0 && T <= 192 && NTW == 6 && S == 1 && tile_mode() != 0;
}

// split-K workspace of the largest plan (0: unsplit); f32: an epilogue of sums;
// aligned: activations on 16-byte boundaries, as a model's own are (those the tile
// kernel takes it takes always: the M-split plans, a microsecond, are not asked for)
static inline size_t gemm_slab_bytes(int T, int N, int K, int epilogue, bool f32 = false, bool aligned = false) {
  const int mtiles = (T + 15) / 16;
  if (mtiles <= 4) {
    const int S = skinny_split(T, N, K, epilogue, true);
    return S > 1 ? (size_t)S * T * ((N + 15) / 16) * 16 * sizeof(float) : 0;
  }
  const int ntiles = (N + 15) / 16 * (epilogue ? 2 : 1);
  int S = 1;
  for (int deferred = f32 ? 1 : 0; deferred <= (epilogue ? 0 : 1); ++deferred) {
    // (of row-major ones: where packed ones go elsewhere, it is with as many slices)
    const bool tiles = K % 32 == 0 && use_tiles(T, N, K, epilogue != 0, false, f32, deferred);
    if (tiles) S = std::max(S, tile_plan(T, N, K, epilogue != 0, f32, deferred).S);
    if (!tiles || !aligned) S = std::max(S, mid_plan(T, N, K, epilogue, deferred).S);
  }
  return S > 1 ? (size_t)S * T * ntiles * 16 * sizeof(float) : 0;
}

// Sum of the S slabs and the epilogue, where no consumer does it.
template <int E>
static hipError_t run_reduce(const float *ws, uint16_t *Y, int T, int N, int ntiles, int S, int yp,
                             float lim, hipStream_t s) {
  const long total = (long)T * ((N + 3) / 4);
  const unsigned blocks = (unsigned)((total + 255) / 256);
#define FFMI_RED(MS)                                                                          \
  hipLaunchKernelGGL((gemm_reduce_kernel<E, MS>), dim3(blocks), dim3(256), 0, s, ws, Y, T, N, \
                     ntiles, S, yp, lim)
  if (S <= 2) FFMI_RED(2);
  else if (S <= 4) FFMI_RED(4);
  else FFMI_RED(8);
#undef FFMI_RED
  return hipGetLastError();
}

template <int E, int MTW, int NTW, int PF>
static hipError_t run_mid(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws,
                          size_t ws_bytes, int T, int N, int K, hipStream_t s,
                          bool xpacked, int yp, int S, Partials *defer, bool nt, int wpitch,
                          float lim) {
  const int KT = K / 32;
  constexpr bool epi = epi_paired<E>;
  const int ntiles = (N + 15) / 16 * (epi ? 2 : 1);
  const size_t wts = w_tile_stride(KT), wks = w_k_stride(wpitch ? wpitch : ntiles);
  const int mtiles = (T + 15) / 16;
  const int mblocks = (mtiles + 4 * MTW - 1) / (4 * MTW);
  const int nblk = (ntiles + NTW - 1) / NTW;
  const size_t need = (size_t)S * T * ntiles * 16 * sizeof(float);
  if (S > 1 && (!ws || ws_bytes < need)) S = 1;  // no workspace: un-split (slower)
  dim3 grid(nblk, S, mblocks);
  static const bool stamp = getenv("FFMI_GEMM_STAMP") != nullptr;
  // unconditional weight loads (ULD) whenever NTW % 4 != 0 (gate/up T = 168:
  // 55.9 -> 51.2 us, qkv 37.2 -> 34.6 us in scripts/gemm_bench.py);
  // FFMI_MID_ULD=0 turns them off (A/B runs)
  static const bool uld = !getenv("FFMI_MID_ULD") || atoi(getenv("FFMI_MID_ULD")) != 0;
  // non-temporal weight loads only where each weight tile has ONE reader
  // (mblocks == 1); prefill blocks re-read every tile from L2 / the MALL
  const bool ntl = nt && mblocks == 1;
#define FFMI_MID2(ST, XPK, U, NL)                                                                  \
  hipLaunchKernelGGL((gemm_mid_kernel<MTW, NTW, PF, E, ST, XPK, U, NL>), grid, dim3(256), 0, s, X, \
                     Wp, Y, ws, T, N, K, KT, ntiles, S, yp, wts, wks, lim)
#define FFMI_MID(ST, XPK)                                     \
  do {                                                        \
    const bool u_ = uld && NTW % 4;                           \
    if (ST) FFMI_MID2(ST, XPK, false, false);                 \
    else if (u_ && ntl) FFMI_MID2(false, XPK, true, true);    \
    else if (u_) FFMI_MID2(false, XPK, true, false);          \
    else if (ntl) FFMI_MID2(false, XPK, false, true);         \
    else FFMI_MID2(false, XPK, false, false);                 \
  } while (0)
  bool done = false;
  if constexpr (E == 0) {
    if (stamp && stamp_buf()) {
      g_stamp_entries = (long)nblk * S * mblocks * 4;
      if (xpacked) FFMI_MID(true, true);
      else FFMI_MID(true, false);
      done = true;
    }
  }
  if constexpr (E < 2) {
    if (!done && !xpacked) {
      FFMI_MID(false, false);
      done = true;
    }
  } else if (!xpacked) {  // (bf16 callers keep their activations packed)
    return hipErrorInvalidValue;
  }
  if (!done) FFMI_MID(false, true);
#undef FFMI_MID
#undef FFMI_MID2
  if (defer) {
    defer->S = 0;
    if ((S > 1 && !epi) || epi_f32<E>) {  // the consumer combines the slabs
      defer->p = ws, defer->S = S, defer->NP = ntiles * 16;
      return hipGetLastError();
    }
  }
  if (S > 1 && !epi_f32<E>) return run_reduce<E>(ws, Y, T, N, ntiles, S, yp, lim, s);
  return hipGetLastError();
}

template <int E>
static hipError_t run_tiles(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws,
                            size_t ws_bytes, int T, int N, int K, hipStream_t s, bool xp, int yp,
                            Partials *defer, bool nt, int wpitch, float lim) {
  constexpr bool paired = epi_paired<E>, f32 = epi_f32<E>;
  const int KT = K / 32, ntiles = (N + 15) / 16 * (paired ? 2 : 1);
  TilePlan p = tile_plan(T, N, K, paired, f32, defer != nullptr && !paired);
  // (fp32 sums without a consumer of slabs, or no room for them: unsplit)
  if ((f32 && !defer) || ws_bytes < (size_t)p.S * T * ntiles * 16 * sizeof(float) || !ws) p.S = 1;
  const size_t wts = w_tile_stride(KT), wks = w_k_stride(wpitch ? wpitch : ntiles);
  static_for<kNumTileForms>([&](auto Fc) {
    constexpr int f = decltype(Fc)::value;
    constexpr TileForm F = kTileForms[f];
    if (p.form != f) return;
    const dim3 grid(p.nbm * p.nbn * p.S), block(F.WR * F.WC * 64);
    if constexpr (F.MI * F.WR == 16)  // (the forms of which one row block holds more than 192 rows)
      if (nt && p.nbm == 1) {
        hipLaunchKernelGGL((gemm_tile_kernel<E, F.MI, F.NJ, F.WR, F.WC, F.NB, true>), grid, block, 0, s, X, Wp, Y,
                           ws, T, N, KT, ntiles, p.nbm, p.S, xp ? 1 : 0, yp, wts, wks, lim);
        return;
      }
    hipLaunchKernelGGL((gemm_tile_kernel<E, F.MI, F.NJ, F.WR, F.WC, F.NB, false>), grid, block, 0, s, X, Wp, Y, ws,
                       T, N, KT, ntiles, p.nbm, p.S, xp ? 1 : 0, yp, wts, wks, lim);
  });
  if (defer && ((p.S > 1 && !paired) || f32)) {
    defer->p = ws, defer->S = p.S, defer->NP = ntiles * 16;
    return hipGetLastError();
  }
  if (p.S > 1 && !f32) return run_reduce<E>(ws, Y, T, N, ntiles, p.S, yp, lim, s);
  return hipGetLastError();
}

// Up to 192 rows in one block, 96 columns a workgroup: the tile kernel with 12 waves
// in the M-split kernel's place, unsplit (the same bits).
template <int E>
static hipError_t run_six(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws, int T, int N, int K,
                          hipStream_t s, int yp, Partials *defer, bool nt, int wpitch, float lim) {
  const int KT = K / 32, ntiles = (N + 15) / 16 * (epi_paired<E> ? 2 : 1);
  const size_t wts = w_tile_stride(KT), wks = w_k_stride(wpitch ? wpitch : ntiles);
  const dim3 grid((ntiles + 5) / 6), block(768);
#define FFMI_SIX(MI, NB, NL)                                                                               \
  hipLaunchKernelGGL((gemm_tile_kernel<E, MI, 2, 4, 3, NB, NL>), grid, block, 0, s, X, Wp, Y, ws, T, N, KT, \
                     ntiles, 1, 1, 1, yp, wts, wks, lim)
  if (T <= 128) {
    if (nt) FFMI_SIX(2, 5, true);
    else FFMI_SIX(2, 5, false);
  } else {
    if (nt) FFMI_SIX(3, 4, true);
    else FFMI_SIX(3, 4, false);
  }
#undef FFMI_SIX
  if (defer && epi_f32<E>) defer->p = ws, defer->S = 1, defer->NP = ntiles * 16;
  return hipGetLastError();
}

// E: the epilogue kind.  Kind 4 takes its slab buffer in `ws` (at least
// T * ntiles * 16 floats) and reports it in *defer; without `defer` it runs
// unsplit, [T][ntiles * 16] in `ws`.
template <int E>
static hipError_t launch_gemm_kind(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws,
                       size_t ws_bytes, int T, int N, int K, int epilogue, hipStream_t s,
                       Partials *defer, int wpitch, const FuseArgs *fuse) {
  if (defer) defer->S = 0;
  if (T <= 0) return hipSuccess;
  const int KT = K / 32;
  const int mtiles = (T + 15) / 16;
  const bool xp = (epilogue & FFMI_X_PACKED) != 0;
  // packed output: the width of the packed rows (N, or wider: fuse->y_width)
  const int yp = !(epilogue & FFMI_Y_PACKED) ? 0 : fuse && fuse->y_width ? fuse->y_width : N;
  const bool nt = (epilogue & FFMI_W_STREAM) != 0;
  constexpr int paired = epi_paired<E> ? 1 : 0;
  const float lim = fuse ? fuse->limit : 0.f;
  if (epi_f32<E> && (!ws || ws_bytes < (size_t)T * ((N + 15) / 16) * 16 * sizeof(float)))
    return hipErrorInvalidValue;
  if ((xp && K % 32) || (yp && (N % 32 || yp % 32 || yp < N))) return hipErrorInvalidValue;
  if constexpr (E < 2)
  if (fuse && fuse->kind) {
    // producer: row-major residual out, plain epilogue; consumer: X is the
    // residual, K = the norm width; both unsplit, T <= 16
    if (mtiles > 1 || N % 16 || K % 32) return hipErrorInvalidValue;
    if (fuse->kind == 1 && (paired || yp || !fuse->res_in || !fuse->ss_out || (fuse->res_packed && N % 32)))
      return hipErrorInvalidValue;
    if (fuse->kind == 2 && (!fuse->ss_in || !fuse->wnorm || fuse->nss <= 0 || fuse->nss > 256 || K > 4096))
      return hipErrorInvalidValue;
    const int wp = wpitch ? wpitch : (paired ? 2 : 1) * ((N + 15) / 16);
    if (fuse->kind == 1) return dispatch_fused<1>(X, Wp, Y, T, N, K, KT, paired, s, xp, yp, nt, wp, *fuse);
    return dispatch_fused<2>(X, Wp, Y, T, N, K, KT, paired, s, xp, yp, nt, wp, *fuse);
  }
  if constexpr (E == 4 || E == 5)
  if (fuse && fuse->kind) {
    const int ntiles = (N + 15) / 16, wp = wpitch ? wpitch : (paired ? 2 : 1) * ntiles;
    const bool producer = fuse->kind == 3;
    if (mtiles > 1 || !xp || (producer ? E != 4 || N % 32 || !fuse->x || (fuse->w32 && (!fuse->hb || !fuse->ss_out))
                                       : fuse->kind != 4 || !fuse->ss_in || fuse->nss < 1 || fuse->nss > 256 ||
                                             fuse->width < 1))
      return hipErrorInvalidValue;
    if constexpr (E == 5) {
      return run<1, 2, 4, 8, E, 4>(X, Wp, Y, ws, T, N, K, KT, 2 * ntiles, 1, s, 1, yp, nt, wp, *fuse);
    } else {
      // (dispatch_nt's forms)
      int S = producer ? 1 : skinny_split(T, N, K, paired, defer != nullptr);
      if (S > 1 && ws_bytes < (size_t)S * T * ntiles * 16 * sizeof(float)) S = 1;
      const bool eight = ntiles < 512 && (KT + S - 1) / S >= 64 && !nt;
      hipError_t e;
      if (producer && eight) e = run<1, 1, 8, 8, E, 3>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, 1, 0, nt, wp, *fuse);
      else if (producer) e = run<1, 1, 4, 8, E, 3>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, 1, 0, nt, wp, *fuse);
      else if (eight) e = run<1, 1, 8, 8, E, 4>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, 1, 0, nt, wp, *fuse);
      else e = run<1, 1, 4, 8, E, 4>(X, Wp, Y, ws, T, N, K, KT, ntiles, S, s, 1, 0, nt, wp, *fuse);
      if (!producer && defer && e == hipSuccess) defer->p = ws, defer->S = S, defer->NP = ntiles * 16;
      return e;
    }
  }
  // (the tile kernel's copies to LDS are of 16 bytes)
  const bool aligned = (((uintptr_t)X | (uintptr_t)Wp) & 15) == 0;
  if (mtiles > 4 && K % 32 == 0 && aligned && (xp || E < 2) &&
      use_tiles(T, N, K, paired, xp, epi_f32<E>, defer != nullptr && !paired))
    return run_tiles<E>(X, Wp, Y, ws, ws_bytes, T, N, K, s, xp, yp, defer, nt, wpitch, lim);
  if (mtiles > 4) {
    const MidPlan p = mid_plan(T, N, K, paired, defer != nullptr && !paired);
#define FFMI_RUN(M, NW) \
  return run_mid<E, M, NW, 4>(X, Wp, Y, ws, ws_bytes, T, N, K, s, xp, yp, SM, defer, nt, wpitch, lim)
    int SM = epi_f32<E> && !defer ? 1 : p.S;
    if (SM > 1 && (!ws || ws_bytes < (size_t)SM * T * ((N + 15) / 16 * 16 << paired) * sizeof(float)))
      SM = 1;  // no workspace: un-split (slower)
    if (takes_six(T, K, p.NTW, SM, xp && aligned))
      return run_six<E>(X, Wp, Y, ws, T, N, K, s, yp, defer, nt, wpitch, lim);
    if (p.MTW == 3) {
      if (p.NTW == 2) FFMI_RUN(3, 2);
      if (p.NTW == 4) FFMI_RUN(3, 4);
      if (p.NTW == 16) FFMI_RUN(3, 16);
      if (p.NTW == 12) FFMI_RUN(3, 12);
      if (p.NTW == 6) FFMI_RUN(3, 6);
      FFMI_RUN(3, 8);
    }
    if (p.NTW == 2) FFMI_RUN(2, 2);
    if (p.NTW == 4) FFMI_RUN(2, 4);
    if (p.NTW == 16) FFMI_RUN(2, 16);
    if (p.NTW == 12) FFMI_RUN(2, 12);
    if (p.NTW == 6) FFMI_RUN(2, 6);
    FFMI_RUN(2, 8);
#undef FFMI_RUN
  }
  const int xi = xp ? 1 : 0;
  const FuseArgs fz = fuse ? *fuse : FuseArgs();
  int S = skinny_split(T, N, K, paired, defer != nullptr);
  const size_t need = (size_t)S * T * ((N + 15) / 16) * 16 * sizeof(float);
  if (S > 1 && (!ws || ws_bytes < need)) S = 1;
  hipError_t e;
  if (mtiles <= 1) e = dispatch_nt<E, 1, 8>(X, Wp, Y, ws, T, N, K, KT, S, s, xi, yp, nt, wpitch, fz);
  else if (mtiles <= 2) e = dispatch_nt<E, 2, 8>(X, Wp, Y, ws, T, N, K, KT, S, s, xi, yp, nt, wpitch, fz);
  else if (mtiles <= 3) {
    // 33 to 48 rows, cold, as four row tiles, three in batches of four k-steps and of eight:
    // 6432 x 2048 11.5 us, 11.3, 10.8; 2048 x 4096 10.7, 10.5, 10.0; 768 x 3072 (fewer than eight k-steps a
    // wave) 6.7, 5.9, 6.8; two tiles a workgroup: 32000 x 4096 57.3, 53.5, 54.5, gate and up of
    // 11008 x 4096 42.2, 39.1, 40.1.  A rest of a batch of eight is worth a batch (a wave's k-steps
    // in brackets): 3072 x 1536 (12) 5.7, 5.4, 6.1; 6144 x 3072 (12) 17.3, 16.0, 17.5; 6144 x 5632
    // (22) 26.0, 23.9, 27.7.
    const int waves = (KT + S - 1) / S >= 64 && !nt ? 8 : 4, mine = ((KT + S - 1) / S + waves - 1) / waves;
    const bool eight = !paired && (N + 15) / 16 < 512 && mine >= 8 && mine % 8 == 0;
    if (eight) e = dispatch_nt<E, 3, 8>(X, Wp, Y, ws, T, N, K, KT, S, s, xi, yp, nt, wpitch, fz);
    else e = dispatch_nt<E, 3, 4>(X, Wp, Y, ws, T, N, K, KT, S, s, xi, yp, nt, wpitch, fz);
  }
  else e = dispatch_nt<E, 4, 4>(X, Wp, Y, ws, T, N, K, KT, S, s, xi, yp, nt, wpitch, fz);
  if ((S > 1 || epi_f32<E>) && defer && e == hipSuccess) defer->p = ws, defer->S = S, defer->NP = (N + 15) / 16 * 16;
  return e;
}

}  // namespace ffmi
