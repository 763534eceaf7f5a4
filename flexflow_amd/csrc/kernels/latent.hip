// latent.hip -- latent attention over a paged cache (latent.h).
#include <algorithm>
#include <type_traits>

#include "device_util.h"
#include "latent.h"

namespace ffmi {

// ---------------------------------------------------------------------------
// latent store: one wave per token
// ---------------------------------------------------------------------------
template <class E>
__device__ __forceinline__ void latent_store_token(const PagedToken &tk, const E *d, const float *w,
                                                   E *cache, int rank, int n, float eps) {
  const int lane = threadIdx.x & 63;
  float ss = 0.f;
  for (int i = lane; i < rank; i += 64) {
    const float v = ld_elem(d + i);
    ss = fmaf(v, v, ss);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float r = inv_rms(ss, n, eps);
  E *dst = cache + (size_t)tk.row * rank;
  for (int i = lane; i < rank; i += 64) st_elem(dst + i, ld_elem(d + i) * r * w[i]);
}

__global__ __launch_bounds__(256) void latent_store_f32_kernel(const PagedToken *__restrict__ tok,
                                                               int T, LatentStore st) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  latent_store_token(tok[t], (const float *)st.d + (size_t)t * st.ldd, st.w, (float *)st.cache,
                     st.rank, st.n, st.eps);
}
hipError_t launch_latent_store_f32(const char *blob, int off_tokens, int T, const LatentStore &st,
                                   hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(latent_store_f32_kernel, dim3((T + 3) / 4), dim3(256), 0, s,
                     reinterpret_cast<const PagedToken *>(blob + off_tokens), T, st);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// per-head products (bf16 MFMA): Y[t][h][n] = sum_k X[t][h][k] W_h[n][k]
// ---------------------------------------------------------------------------
// W_h tile-major: block (h, nt, kt) of 16 x 32 at ((h * NTt + nt) * KT + kt) *
// 512.  Four waves, WM of them over row groups of MT tiles, 4 / WM over groups
// of NT weight tiles.  D = W . X^T: a lane holds four consecutive columns of
// one row.
struct HgDev {
  const uint16_t *X, *W, *gate;
  uint16_t *Y;
  int T, heads, KT, NTt, ldx, ldg, packed;
  int gx, gz;  // weight-tile groups, row groups of the launch
};
template <int MT, int NT, int WM>
__device__ __forceinline__ void head_gemm_block(const HgDev &a, int b) {
  constexpr int WN = 4 / WM;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, l15 = lane & 15;
  const int bx = b % a.gx, h = (b / a.gx) % a.heads, bz = b / (a.gx * a.heads);
  const int nt0 = (bx * WN + wave % WN) * NT;
  const int m0 = (bz * WM + wave / WN) * MT * 16;
  if (nt0 >= a.NTt || m0 >= a.T) return;
  const int K = a.KT * 32;
  const uint16_t *xr[MT], *wr[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    xr[i] = a.X + (size_t)min(m0 + i * 16 + l15, a.T - 1) * a.ldx + (size_t)h * K + 8 * g;
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wr[j] = a.W + ((size_t)h * a.NTt + min(nt0 + j, a.NTt - 1)) * a.KT * 512 + lane * 8;
  f4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = MT * NT >= 8 ? 2 : 4;  // k-steps of loads issued ahead of their MFMAs
  for (int k0 = 0; k0 < a.KT; k0 += U) {
    bf8 x[U][MT], w[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u, a.KT - 1);
#pragma unroll
      for (int j = 0; j < NT; ++j) w[u][j] = *reinterpret_cast<const bf8 *>(wr[j] + (size_t)k * 512);
#pragma unroll
      for (int i = 0; i < MT; ++i) x[u][i] = *reinterpret_cast<const bf8 *>(xr[i] + k * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u < a.KT)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][j], x[u][i], acc[i][j], 0, 0, 0);
  }
  const int N = a.NTt * 16, Yw = a.heads * N;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + i * 16 + l15;
    if (m >= a.T) continue;
    float sc = 1.f;
    if (a.gate) sc = __fdiv_rn(1.0f, 1.0f + expf(-bf2f(a.gate[(size_t)m * a.ldg + h])));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (nt0 + j >= a.NTt) continue;
      const int n = h * N + (nt0 + j) * 16 + 4 * g;
      const f4 v = acc[i][j];
      const uint2 o = make_uint2(f2bf(v[0] * sc) | ((uint32_t)f2bf(v[1] * sc) << 16),
                                 f2bf(v[2] * sc) | ((uint32_t)f2bf(v[3] * sc) << 16));
      *reinterpret_cast<uint2 *>(a.Y + (a.packed ? act_packed_off(m, n, Yw) : (size_t)m * Yw + n)) = o;
    }
  }
}

template <int MT, int NT, int WM>
__global__ __launch_bounds__(256) void latent_prep_kernel(const PagedToken *__restrict__ tok,
                                                          HgDev a, int nprod, LatentStore st) {
  if ((int)blockIdx.x < nprod) {
    head_gemm_block<MT, NT, WM>(a, blockIdx.x);
    return;
  }
  const int t = (blockIdx.x - nprod) * 4 + (threadIdx.x >> 6);
  if (t >= a.T) return;
  latent_store_token(tok[t], (const uint16_t *)st.d + (size_t)t * st.ldd, st.w,
                     (uint16_t *)st.cache, st.rank, st.n, st.eps);
}

// More than 128 rows: a workgroup takes 128 rows and 128 columns of a head, its rows through
// LDS in chunks of 64 k, two of them and a chunk of weights on their way.  Read as they lie,
// rows sent the lanes of a load to 16 places, which the L1 serves one after another,
// and two k-steps of loads were all that was under way.  A row's eight 16-byte pieces lie
// exchanged by the row's number; row-major outputs go through LDS as well and leave as
// whole lines.  A head's workgroups share an XCD where heads are a multiple of 8: its
// weights are read from memory once.  1024 rows, 32 heads: K = 128, N = 512 with the latents'
// store 25 -> 21 us, K = 512, N = 128 21 -> 14.
// Up to two chunks of k (KC <= 2) it is a chain of waits, and workgroups side by side are what
// hides them: one chunk's weights in registers at a time leave room for four on a CU instead of
// two (126 registers, 176 before; two and a half rounds of the 1280 before), and the latents'
// workgroups go first instead of behind the last products: 20.3 -> 16.9 us.
__device__ __forceinline__ int prep_turn(int row) { return (row >> 1 & 3) << 1 | (row >> 3 & 1); }
template <int KC>
__device__ __forceinline__ void head_gemm_tile(const HgDev &a, int b, uint16_t *sh) {
  const int lane = threadIdx.x & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = b % a.heads, rest = b / a.heads, nt0 = (rest % a.gx) * 8, m0 = (rest / a.gx) * 128;
  const int wm = wave >> 1, wn = wave & 1, K = KC * 64;
  const uint16_t *x = a.X + (size_t)h * K;
  auto copy = [&](int c) {  // 4 KiB of the chunk's 16 (8 rows a copy)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave * 4 + i) * 8 + (lane >> 3), piece = (lane ^ prep_turn(row)) & 7;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void *)(x + (size_t)min(m0 + row, a.T - 1) * a.ldx + c * 64 + piece * 8),
          (__attribute__((address_space(3))) void *)(sh + c * 8192 + (wave * 4 + i) * 512), 16, 0, 0);
    }
  };
  const uint16_t *w0[4];  // (the wave's; a lane's 16 bytes are lane * 8 on)
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w0[j] = a.W + ((size_t)h * a.NTt + min(nt0 + wn * 4 + j, a.NTt - 1)) * a.KT * 512;
  constexpr int WB = KC <= 2 ? 1 : 2;
  bf8 w[WB][2][4];
  auto weights = [&](int c) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) w[c % WB][k][j] = *reinterpret_cast<const bf8 *>(w0[j] + (2 * c + k) * 512 + lane * 8);
  };
  f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  copy(0);
  if (KC > 1 && WB > 1) copy(1);
  weights(0);
  if (KC > 1 && WB == 1) copy(1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    if (c + 2 < KC) copy(c + 2);
    if (WB > 1 && c + 1 < KC) weights(c + 1);
    if (WB == 1 && c > 0) weights(c);
    __builtin_amdgcn_sched_barrier(0);
    // chunk c has landed, what was just asked for may be under way: s_waitcnt vmcnt
    if (c + 2 < KC) __builtin_amdgcn_s_waitcnt(0x0f70 | 12);
    else if (c + 1 < KC) __builtin_amdgcn_s_waitcnt(0x0f70 | (WB > 1 ? 8 : 4));
    else __builtin_amdgcn_s_waitcnt(0x0f70);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint16_t *xr = sh + c * 8192 + (wm * 64 + l15) * 64;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      bf8 xf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        xf[i] = *reinterpret_cast<const bf8 *>(xr + i * 1024 + ((4 * k + g) ^ prep_turn(l15)) * 8);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c % WB][k][j], xf[i], acc[i][j], 0, 0, 0);
    }
  }
  const int N = a.NTt * 16, Yw = a.heads * N, n0 = nt0 + wn * 4;  // (column tiles)
  __syncthreads();
  uint16_t *mine = sh + wave * 4096;  // 64 rows x 64 columns of this wave, pieces exchanged
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + wm * 64 + i * 16 + l15;
    float sc = 1.f;
    if (a.gate) sc = __fdiv_rn(1.0f, 1.0f + expf(-bf2f(a.gate[(size_t)min(m, a.T - 1) * a.ldg + h])));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f4 v = acc[i][j];
      const uint2 o = make_uint2(f2bf(v[0] * sc) | ((uint32_t)f2bf(v[1] * sc) << 16),
                                 f2bf(v[2] * sc) | ((uint32_t)f2bf(v[3] * sc) << 16));
      if (a.packed) {
        if (m < a.T && n0 + j < a.NTt)
          *reinterpret_cast<uint2 *>(a.Y + act_packed_off(m, h * N + (n0 + j) * 16 + 4 * g, Yw)) = o;
      } else {
        const int piece = (2 * j + (g >> 1)) ^ prep_turn(l15);
        *reinterpret_cast<uint2 *>(mine + (i * 16 + l15) * 64 + piece * 8 + 4 * (g & 1)) = o;
      }
    }
  }
  if (a.packed) return;
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's own writes
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = i * 8 + (lane >> 3), m = m0 + wm * 64 + row, p = lane & 7;
    const uint4 v = *reinterpret_cast<const uint4 *>(mine + row * 64 + ((p ^ prep_turn(row & 15)) * 8));
    if (m < a.T && n0 + (p >> 1) < a.NTt)
      *reinterpret_cast<uint4 *>(a.Y + (size_t)m * Yw + h * N + n0 * 16 + p * 8) = v;
  }
}
template <int KC>
__global__ __launch_bounds__(256, KC <= 2 ? 4 : 1) void latent_prep_tile_kernel(const PagedToken *__restrict__ tok, HgDev a,
                                                               int nprod, LatentStore st) {
  __shared__ __attribute__((aligned(16))) uint16_t sh[(KC < 2 ? 2 : KC) * 8192];
  const int nst = (int)gridDim.x - nprod;
  if ((int)blockIdx.x >= nst) {
    head_gemm_tile<KC>(a, blockIdx.x - nst, sh);
    return;
  }
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.T) return;
  latent_store_token(tok[t], (const uint16_t *)st.d + (size_t)t * st.ldd, st.w,
                     (uint16_t *)st.cache, st.rank, st.n, st.eps);
}

static hipError_t run_prep(const PagedToken *tok, const LatentStore &st, const HeadGemm &hg,
                           hipStream_t s) {
  if (hg.T <= 0) return hipSuccess;
  if (hg.K % 32 || hg.N % 32 || hg.ldx % 8) return hipErrorInvalidValue;
  HgDev a;
  a.X = (const uint16_t *)hg.X, a.W = (const uint16_t *)hg.W, a.gate = (const uint16_t *)hg.gate;
  a.Y = (uint16_t *)hg.Y;
  a.T = hg.T, a.heads = hg.heads, a.KT = hg.K / 32, a.NTt = hg.N / 16, a.ldx = hg.ldx;
  a.ldg = hg.ldg, a.packed = hg.packed ? 1 : 0;
  const int nst = st.cache ? (hg.T + 3) / 4 : 0;
#define FFMI_PREP(MT, NT, WM)                                                                   \
  do {                                                                                          \
    a.gx = (a.NTt + (4 / WM) * NT - 1) / ((4 / WM) * NT);                                       \
    a.gz = (hg.T + WM * MT * 16 - 1) / (WM * MT * 16);                                          \
    const int np = a.gx * a.heads * a.gz;                                                       \
    hipLaunchKernelGGL((latent_prep_kernel<MT, NT, WM>), dim3(np + nst), dim3(256), 0, s, tok, a, \
                       np, st);                                                                 \
  } while (0)
// (widths that heads and latents have; their rows have to fit the LDS)
#define FFMI_PREP_TILE(KC)                                                                      \
  do {                                                                                          \
    a.gx = (a.NTt + 7) / 8, a.gz = (hg.T + 127) / 128;                                          \
    const int np = a.gx * a.heads * a.gz;                                                       \
    hipLaunchKernelGGL((latent_prep_tile_kernel<KC>), dim3(np + nst), dim3(256), 0, s, tok, a, np, st); \
  } while (0)
  if (hg.T <= 16) FFMI_PREP(1, 1, 1);
  else if (hg.T <= 32) FFMI_PREP(2, 1, 1);
  else if (hg.T <= 128) FFMI_PREP(2, 2, 1);
  else if (hg.K == 64) FFMI_PREP_TILE(1);
  else if (hg.K == 128) FFMI_PREP_TILE(2);
  else if (hg.K == 192) FFMI_PREP_TILE(3);
  else if (hg.K == 256) FFMI_PREP_TILE(4);
  else if (hg.K == 384) FFMI_PREP_TILE(6);
  else if (hg.K == 512) FFMI_PREP_TILE(8);
  else FFMI_PREP(4, 4, 2);
#undef FFMI_PREP_TILE
#undef FFMI_PREP
  return hipGetLastError();
}
hipError_t launch_latent_prep(const char *blob, int off_tokens, const LatentStore &st,
                              const HeadGemm &hg, hipStream_t s) {
  return run_prep(reinterpret_cast<const PagedToken *>(blob + off_tokens), st, hg, s);
}
hipError_t launch_head_gemm(const HeadGemm &hg, hipStream_t s) {
  return run_prep(nullptr, LatentStore(), hg, s);
}

// fp32: W_h as [K][N] row-major, one workgroup per (token, head)
__global__ __launch_bounds__(256) void head_gemm_f32_kernel(const float *__restrict__ X,
                                                            const float *__restrict__ W,
                                                            const float *__restrict__ gate,
                                                            float *__restrict__ Y, int heads, int K,
                                                            int N, int ldx, int ldg) {
  const int t = blockIdx.x, h = blockIdx.y;
  const float *x = X + (size_t)t * ldx + (size_t)h * K, *w = W + (size_t)h * K * N;
  const float sc =
      gate ? __fdiv_rn(1.0f, 1.0f + expf(-gate[(size_t)t * ldg + h])) : 1.0f;
  for (int n = threadIdx.x; n < N; n += 256) {
    float acc = 0.f;
    for (int k = 0; k < K; ++k) acc = fmaf(x[k], w[(size_t)k * N + n], acc);
    Y[((size_t)t * heads + h) * N + n] = acc * sc;
  }
}
hipError_t launch_head_gemm_f32(const HeadGemm &hg, hipStream_t s) {
  if (hg.T <= 0) return hipSuccess;
  hipLaunchKernelGGL(head_gemm_f32_kernel, dim3(hg.T, hg.heads), dim3(256), 0, s,
                     (const float *)hg.X, (const float *)hg.W, (const float *)hg.gate,
                     (float *)hg.Y, hg.heads, hg.K, hg.N, hg.ldx, hg.ldg);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// attention over the pages, MFMA form
// ---------------------------------------------------------------------------
// Up to 32 rows (RT = 1, 2): one workgroup of eight waves, up to RT * 16 rows against a
// range of 64-token pages.  Scores S^T = C . Q'^T (lane: 4 keys of one row), outputs O^T = C^T .
// P^T with C^T read from the row-major page in LDS by the transposing LDS load;
// the k order of the second product is the key order the scores already have
// in the lanes (16-lane group g: keys 4g..4g+3 and 16+4g..).
//   scores:  wave = (16-key tile, row tile); RT == 1: four waves only
//   outputs: each wave an eighth of the latent's columns, all rows
// Softmax state in fp32, base-2 exponents; weights meet the second product in
// bf16, the sums take them unrounded.
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
constexpr int kRankPad = 8;  // LDS row padding (elements)

template <int RC, int RT>
__global__ __launch_bounds__(512) void latent_attn_kernel(
    const char *__restrict__ blob, int off_blocks, const uint16_t *__restrict__ Q,
    const uint16_t *__restrict__ cache, uint16_t *__restrict__ O, float *__restrict__ slabs,
    float *__restrict__ ml, int heads, float scale_log2) {
  constexpr int R = RC * 64, KS = RC * 2, LDC = R + kRankPad;
  constexpr int NT = RC * 4, DT = (NT + 7) / 8;  // column tiles: all, of a wave's outputs
  constexpr int LDP = kPageTokens + 8;
  __shared__ __attribute__((aligned(16))) uint16_t sC[2][64 * LDC];
  __shared__ __attribute__((aligned(16))) uint16_t sP[RT * 16 * LDP];
  __shared__ float sM[4][RT * 16], sL[4][RT * 16];
  const PagedBlock bk = reinterpret_cast<const PagedBlock *>(blob + off_blocks)[blockIdx.x];
  if (bk.nrows <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave & 3, wr = wave >> 2;
  const bool scoring = RT > 1 || wr == 0;
  const int32_t *table = reinterpret_cast<const int32_t *>(blob) + bk.table;

  // the next page through registers, RC 16-byte chunks per thread
  auto page_at = [&](int i0) {
    return cache + (size_t)(i0 == 0 ? bk.page0 : table[bk.tile0 + i0]) * (64 * R);
  };
  u4 pre[RC];
  auto fetch = [&](int i0) {
    const uint16_t *page = page_at(i0);
#pragma unroll
    for (int i = 0; i < RC; ++i) pre[i] = *reinterpret_cast<const u4 *>(page + (tid + i * 512) * 8);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < RC; ++i) {
      const int c = tid + i * 512;
      *reinterpret_cast<u4 *>(&sC[buf][(c / (R / 8)) * LDC + (c % (R / 8)) * 8]) = pre[i];
    }
  };
  fetch(0);
  // this wave's rows of Q' as B operands (rows past the block re-read its last)
  bf8 q[KS];
  const int qr = min(wr * 16 + l15, bk.nrows - 1);
  const uint16_t *qp = Q + (size_t)(bk.row0 + qr) * R + 8 * g;
#pragma unroll
  for (int k = 0; k < KS; ++k) q[k] = *reinterpret_cast<const bf8 *>(qp + k * 32);
  const int qpos = bk.pos0 + (bk.row0 + qr - bk.seg_row) / heads;
  f4 acc[RT][DT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[i][d] = f4{0.f, 0.f, 0.f, 0.f};
  float m[RT], l = 0.f;
#pragma unroll
  for (int i = 0; i < RT; ++i) m[i] = -1e30f;
  stage(0);
  if (bk.ntiles > 1) fetch(1);
  __syncthreads();
  for (int it = 0; it < bk.ntiles; ++it) {
    const uint16_t *C = sC[it & 1];
    f4 s;
    if (scoring) {
      // two chains (even / odd k-steps)
      f4 s2 = f4{0.f, 0.f, 0.f, 0.f};
      s = s2;
#pragma unroll
      for (int ks = 0; ks < KS; ks += 2) {
        const uint16_t *cr = &C[(wk * 16 + l15) * LDC + ks * 32 + 8 * g];
        const bf8 c0 = *reinterpret_cast<const bf8 *>(cr), c1 = *reinterpret_cast<const bf8 *>(cr + 32);
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c0, q[ks], s, 0, 0, 0);
        s2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c1, q[ks + 1], s2, 0, 0, 0);
      }
      // scale, mask, this wave's maximum of every row
      const int key0 = (bk.tile0 + it) * 64 + wk * 16 + 4 * g;
      float mx = -1e30f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = key0 + e <= qpos ? (s[e] + s2[e]) * scale_log2 : -INFINITY;
        s[e] = v;
        mx = fmaxf(mx, v);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (g == 0) sM[wk][wr * 16 + l15] = mx;
    }
    __syncthreads();
    float alpha[RT];
    bool moved = false;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      float mn = m[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) mn = fmaxf(mn, sM[k][i * 16 + l15]);
      alpha[i] = __builtin_amdgcn_exp2f(m[i] - mn);
      moved |= mn != m[i];
      m[i] = mn;
    }
    if (scoring) {
      const float mi = RT > 1 && wr ? m[RT - 1] : m[0];
      const float ai = RT > 1 && wr ? alpha[RT - 1] : alpha[0];
      float p[4], sum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = __builtin_amdgcn_exp2f(s[e] - mi);
        sum += p[e];
      }
      *reinterpret_cast<uint2 *>(&sP[(wr * 16 + l15) * LDP + wk * 16 + 4 * g]) =
          make_uint2(f2bf(p[0]) | ((uint32_t)f2bf(p[1]) << 16), f2bf(p[2]) | ((uint32_t)f2bf(p[3]) << 16));
      l = l * ai + sum;
    }
    if (it + 1 < bk.ntiles) {
      stage((it + 1) & 1);  // (last read by the outputs of tile it - 1)
      if (it + 2 < bk.ntiles) fetch(it + 2);
    }
    __syncthreads();
    if (__any(moved))
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[i][d] *= alpha[i];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s8 p[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const uint16_t *pr = &sP[(i * 16 + l15) * LDP + kb * 32 + 4 * g];
        const s4 lo = *reinterpret_cast<const s4 *>(pr), hi = *reinterpret_cast<const s4 *>(pr + 16);
        p[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        if (NT % 8 && wave * DT + d >= NT) continue;
        const uint16_t *cr =
            &C[(kb * 32 + 4 * g + (l15 >> 2)) * LDC + (wave * DT + d) * 16 + 4 * (l15 & 3)];
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s4 *)(cr));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s4 *)(cr + 16 * LDC));
        const bf8 a = __builtin_bit_cast(
            bf8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int i = 0; i < RT; ++i)
          acc[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf8, p[i]),
                                                              acc[i][d], 0, 0, 0);
      }
    }
  }
  if (scoring) {
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) sL[wk][wr * 16 + l15] = l;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    float sum = sL[0][i * 16 + l15];
#pragma unroll
    for (int k = 1; k < 4; ++k) sum += sL[k][i * 16 + l15];
    const int r = i * 16 + l15;
    if (r >= bk.nrows) continue;
    if (bk.slot >= 0) {
      const size_t pr = (size_t)bk.slot * (RT * 16) + r;
#pragma unroll
      for (int d = 0; d < DT; ++d)
        if (NT % 8 == 0 || wave * DT + d < NT)
          *reinterpret_cast<f4 *>(slabs + pr * R + (wave * DT + d) * 16 + 4 * g) = acc[i][d];
      if (wave == 0 && g == 0) ml[pr * 2] = m[i], ml[pr * 2 + 1] = sum;
    } else {
      const float inv = __fdiv_rn(1.0f, sum);
      uint16_t *o = O + (size_t)(bk.row0 + r) * R + wave * DT * 16 + 4 * g;
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        if (NT % 8 && wave * DT + d >= NT) continue;
        const f4 v = acc[i][d] * inv;
        *reinterpret_cast<uint2 *>(o + d * 16) =
            make_uint2(f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                       f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
      }
    }
  }
}

// More than 32 rows (prompts), 64 a block.  Half pages of 32 tokens: waves 0..3 copy half
// pages to LDS, score 16 rows each against all 32 keys of a half (so that a row's maximum
// needs no other wave) and leave the weights in LDS; waves 4..7 add a half's outputs up, a
// quarter of the latent's columns each, one half behind.  A SIMD has a wave of either kind:
// one's products run beside the other's exponentials and reads.  One barrier a half; two
// halves are on their way and one in each kind's hands.  A workgroup takes block after
// block, the next one's rows of Q' and first half copied while this one's last halves are
// added up, its outputs stored beside the next one's first scores.
// What bounds it: the LDS (each scoring wave reads the whole half: 128 of 210 KiB a half
// at rank 512) at 2300 cycles a half, then Q' and O (64 KiB each a block).  Before, all
// eight waves took turns (scores, barrier, weights, barrier, outputs, barrier a page), Q'
// was read as it lies (16 rows a load, 256 loads) and the compiler waited for the next page
// as soon as it was asked for.  32 heads, rank 512, prompt steps of 1024, 1024 and 620
// tokens: 70 -> 53 us a launch, of which a page of 64 rows takes 2.2.
// A half's rows lie one after another, the 16-byte pieces of each 256 bytes (of 128 where rows
// are whole 128s, so that every other row starts at the other half) exchanged by the
// row's number: a read of scores takes one piece of 16 rows, of outputs two of 8.
template <int RC>
constexpr int kLatentPieces = RC % 2 == 0 ? 16 : 8;
template <int RC>
__device__ __forceinline__ int latent_turn(int row) {
  return RC % 2 == 0 ? (row & 7) << 1 | (row >> 3 & 1) : (row >> 1 & 3) << 1 | (row >> 3 & 1);
}
template <int RC>
constexpr int kLatentWide = RC <= 4 ? 2 : 1;  // workgroups of a CU, by their LDS
template <int RC>
__global__ __launch_bounds__(512) void latent_attn_wide_kernel(
    const char *__restrict__ blob, int off_blocks, int num_blocks, const uint16_t *__restrict__ Q,
    const uint16_t *__restrict__ cache, uint16_t *__restrict__ O, float *__restrict__ slabs,
    float *__restrict__ ml, int heads, float scale_log2) {
  constexpr int R = RC * 64, KS = RC * 2, H = 32;  // H: tokens of a half
  constexpr int PP = kLatentPieces<RC>, KP = PP / 4, CP = PP / 2;  // pieces, k-steps, column tiles of an exchange
  constexpr int LDP = H + 8;
  // (one array: of several the compiler knows which one a copy writes, and waits for all
  // copies under way before it reads that)
  __shared__ __attribute__((aligned(16))) uint16_t sh[4 * H * R + 2 * 64 * LDP + 2 * (2 * 64 + 2 * 64)];
  uint16_t *sP = sh + 4 * H * R;                                // [half & 1][64][LDP]
  float *sA = reinterpret_cast<float *>(sP + 2 * 64 * LDP);     // [half & 1][64]: what the sums so far shrink by
  float *sM = sA + 2 * 64, *sL = sM + 64;                       // maximum and sum of a row, at a block's end
  const PagedBlock *blocks = reinterpret_cast<const PagedBlock *>(blob + off_blocks);
  const int lane = threadIdx.x & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // this workgroup's k-th block (nrows == 0: none): the list, longest first, dealt out back and
  // forth; padding is at its end
  auto block_of = [&](int k) {
    const int i = k * gridDim.x + (k & 1 ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
    PagedBlock bk{};
    if (i < num_blocks) bk = blocks[i];
    return bk;
  };
  // its halves, up to the last position that its last row sees
  auto halves_of = [&](const PagedBlock &bk) {
    const int last = bk.pos0 + (bk.row0 + bk.nrows - 1 - bk.seg_row) / heads - bk.tile0 * 64;
    return min(2 * bk.ntiles, last / H + 1);
  };
  // a barrier that leaves copies to LDS and stores under way
  auto meet = [] {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  PagedBlock bk = block_of(0);
  if (bk.nrows <= 0) return;
  if (wave < 4) {
    const int32_t *words = reinterpret_cast<const int32_t *>(blob);
    // rows 0 .. 31 (rows past `most`: that one again) to buffer buf & 3, this wave's quarter
    auto copy = [&](const uint16_t *src, int buf, int most) {
#pragma unroll
      for (int i = 0; i < RC; ++i) {
        const int n = (wave * RC + i) * 64 + lane, row = n / (8 * RC), p = n % (8 * RC);
        const int piece = (p & -PP) | ((p ^ latent_turn<RC>(row)) & (PP - 1));
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void *)(src + (size_t)min(row, most) * R + piece * 8),
            (__attribute__((address_space(3))) void *)(sh + (buf & 3) * H * R + (wave * RC + i) * 512), 16, 0, 0);
      }
    };
    auto copy_rows = [&](const PagedBlock &b, int part, int buf) {  // 32 rows of Q'
      copy(Q + (size_t)(b.row0 + min(part * H, b.nrows - 1)) * R, buf, max(b.nrows - 1 - part * H, 0));
    };
    auto copy_half = [&](int h, int page, int buf) { copy(cache + ((size_t)page * 64 + (h & 1) * H) * R, buf, H - 1); };
    // s_waitcnt vmcnt(RC) (the last stage asked for may still be under way) or vmcnt(0)
    auto wait = [](bool more) {
      if (more) __builtin_amdgcn_s_waitcnt((RC & 15) | 0x0f70 | ((RC >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0f70);
      asm volatile("" ::: "memory");
    };
    // this lane's piece of a k-step
    int at[KP];
#pragma unroll
    for (int i = 0; i < KP; ++i) at[i] = l15 * R + ((4 * i + g) ^ latent_turn<RC>(l15)) * 8;
    auto piece = [&](const uint16_t *rows, int ks) {
      return *reinterpret_cast<const bf8 *>(rows + at[ks % KP] + ks / KP * KP * 32);
    };
    int b0 = 0;  // half 0's buffer; the rows of Q' in the two after half 1's
    copy_rows(bk, 0, 2);
    copy_rows(bk, 1, 3);
    copy_half(0, bk.page0, 0);
    wait(false);
    meet();
    for (int k = 0;; ++k) {
      const PagedBlock nb = block_of(k + 1);
      const bool next = nb.nrows > 0;
      const int nh = halves_of(bk);
      auto page_of = [&](int h) { return h < 2 ? bk.page0 : words[bk.table + bk.tile0 + (min(h, nh - 1) >> 1)]; };
      // The stages in turn: this block's halves, the next one's rows of Q' and its half 0, each
      // in the buffer after the last one's.
      auto stage = [&](int e, int page) {
        if (e < nh) copy_half(e, page, b0 + e);
        else if (next && e < nh + 2) copy_rows(nb, e - nh, b0 + e);
        else if (next && e == nh + 2) copy_half(0, nb.page0, b0 + e);
      };
      auto staged = [&](int e) { return e < nh || (next && e <= nh + 2); };
      stage(1, bk.page0);
      int page = page_of(2);  // of the next half to be asked for: read a half ahead
      bf8 q[KS];              // rows 16 wave + l15 as B operands
      const uint16_t *rows = sh + ((b0 + 2 + (wave >> 1)) & 3) * H * R + (wave & 1) * 16 * R;
#pragma unroll
      for (int i = 0; i < KS; ++i) q[i] = piece(rows, i);
      wait(staged(1));
      meet();
      stage(2, page);
      page = page_of(3);
      const int row = min(wave * 16 + l15, bk.nrows - 1);
      const int see = bk.pos0 + (bk.row0 + row - bk.seg_row) / heads - bk.tile0 * 64 - 4 * g;
      float m = -1e30f, l = 0.f;
      auto score = [&](int h) {
        const uint16_t *C = sh + ((b0 + h) & 3) * H * R;
        // per 16 keys two chains (even / odd k-steps); operands read D steps ahead
        constexpr int D = KS < 8 ? KS : 8;
        f4 s[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) s[t][0] = s[t][1] = f4{0.f, 0.f, 0.f, 0.f};
        bf8 c[D][2];
        auto read = [&](int ks) {
          c[ks % D][0] = piece(C, ks);
          c[ks % D][1] = piece(C + 16 * R, ks);
        };
#pragma unroll
        for (int ks = 0; ks < D; ++ks) read(ks);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < 2; ++t)
            s[t][ks & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[ks % D][t], q[ks], s[t][ks & 1], 0, 0, 0);
          if (ks + D < KS) read(ks + D);
        }
        float v[2][4], mx = m;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[t][e] = h * H + t * 16 + e <= see ? (s[t][0][e] + s[t][1][e]) * scale_log2 : -INFINITY;
            mx = fmaxf(mx, v[t][e]);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float shrink = __builtin_amdgcn_exp2f(m - mx);
        float sum = 0.f;
        uint16_t *P = sP + (((h & 1) * 64) + wave * 16 + l15) * LDP + 4 * g;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          s4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = __builtin_amdgcn_exp2f(v[t][e] - mx);
            sum += x;
            w[e] = (short)f2bf(x);
          }
          *reinterpret_cast<s4 *>(P + t * 16) = w;
        }
        if (g == 0) sA[(h & 1) * 64 + wave * 16 + l15] = shrink;
        l = l * shrink + sum;
        m = mx;
      };
      score(0);
      for (int h = 0; h < nh; ++h) {
        wait(staged(h + 2));  // stage h + 1 has landed
        meet();
        // (its buffer was half h - 1's, whose outputs were added up before the barrier, or Q''s)
        stage(h + 3, page);
        page = page_of(h + 4);
        if (h + 1 < nh) score(h + 1);
      }
      l += __shfl_xor(l, 16);
      l += __shfl_xor(l, 32);
      if (g == 0) sM[wave * 16 + l15] = m, sL[wave * 16 + l15] = l;
      wait(next);  // the next block's rows of Q' have landed
      meet();
      if (!next) return;
      b0 = (b0 + nh + 2) & 3;
      bk = nb;
    }
  }
  const int ct0 = (wave - 4) * RC, trow = 4 * g + (l15 >> 2);
  const int tturn = latent_turn<RC>(trow) ^ ((l15 & 3) >> 1), tbase = trow * R + (l15 & 1) * 4;
  int b0 = 0;
  meet();
  meet();
  for (int k = 0;; ++k) {
    const PagedBlock nb = block_of(k + 1);
    const int nh = halves_of(bk);
    f4 acc[4][RC];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int d = 0; d < RC; ++d) acc[i][d] = f4{0.f, 0.f, 0.f, 0.f};
    for (int h = 0; h < nh; ++h) {
      meet();
      const uint16_t *C = sh + ((b0 + h) & 3) * H * R, *P = sP + (h & 1) * 64 * LDP;
      // 16 columns of 32 tokens, transposed: k order as the weights'
      auto columns = [&](int d) {
        const int ct = ct0 + d;
        const uint16_t *p = C + tbase + ct / CP * CP * 16 + ((2 * (ct % CP)) ^ tturn) * 8;
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)(p));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)(p + 16 * R));
        return __builtin_bit_cast(bf8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      };
      bf8 p[4], a[RC];
      float shrink[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) shrink[i] = sA[(h & 1) * 64 + i * 16 + l15];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t *pr = P + (i * 16 + l15) * LDP + 4 * g;
        const s4 lo = *reinterpret_cast<const s4 *>(pr), hi = *reinterpret_cast<const s4 *>(pr + 16);
        p[i] = __builtin_bit_cast(bf8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int d = 0; d < RC; ++d) a[d] = columns(d);
      __builtin_amdgcn_sched_barrier(0);
      if (__any(shrink[0] != 1.f || shrink[1] != 1.f || shrink[2] != 1.f || shrink[3] != 1.f))
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int d = 0; d < RC; ++d) acc[i][d] *= shrink[i];
#pragma unroll
      for (int d = 0; d < RC; ++d) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d], p[i], acc[i][d], 0, 0, 0);
      }
    }
    meet();
    if (nb.nrows > 0) meet();  // (the next block's scores start beside the stores)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i * 16 + l15;
      if (r >= bk.nrows) continue;
      const float sum = sL[r];
      if (bk.slot >= 0) {
        const size_t pr = (size_t)bk.slot * 64 + r;
#pragma unroll
        for (int d = 0; d < RC; ++d) *reinterpret_cast<f4 *>(slabs + pr * R + (ct0 + d) * 16 + 4 * g) = acc[i][d];
        if (wave == 4 && g == 0) ml[pr * 2] = sM[r], ml[pr * 2 + 1] = sum;
      } else {
        const float inv = __fdiv_rn(1.0f, sum);
        uint16_t *o = O + (size_t)(bk.row0 + r) * R + ct0 * 16 + 4 * g;
#pragma unroll
        for (int d = 0; d < RC; ++d) {
          const f4 v = acc[i][d] * inv;
          *reinterpret_cast<uint2 *>(o + d * 16) =
              make_uint2(f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16), f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
        }
      }
    }
    if (nb.nrows <= 0) return;
    b0 = (b0 + nh + 2) & 3;
    bk = nb;
  }
}

// partials of split blocks, in slot order: one workgroup per row, the slots'
// weights first (one lane each), then the slabs in groups of independent loads
template <int RC>
constexpr int kMergeThreads = RC <= 4 ? 64 : 128;
template <int RC>
__global__ __launch_bounds__(kMergeThreads<RC>) void latent_merge_kernel(
    const char *__restrict__ blob, int off_merges, const float *__restrict__ slabs,
    const float *__restrict__ ml, uint16_t *__restrict__ O, int block_rows) {
  constexpr int R = RC * 64, G = 8;
  const PagedMerge mg = reinterpret_cast<const PagedMerge *>(blob + off_merges)[blockIdx.x];
  const int r = blockIdx.y, lane = threadIdx.x & 63;
  if (r >= mg.nrows) return;
  const size_t row0 = (size_t)mg.slot0 * block_rows + r;
  const int col = threadIdx.x * 4;
  const float *sl = slabs + row0 * R + min(col, R - 4);
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  float M = -1e30f, sum = 0.f;
  constexpr int L = 64;  // slots at a time (every wave works out the same weights)
  for (int s0 = 0; s0 < mg.nslots; s0 += L) {
    const int n = min(L, mg.nslots - s0);
    const size_t mi = (row0 + (size_t)(s0 + min(lane, n - 1)) * block_rows) * 2;
    const float m = lane < n ? ml[mi] : -1e30f, l = lane < n ? ml[mi + 1] : 0.f;
    float mx = m;
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    mx = fmaxf(mx, M);
    const float a = __builtin_amdgcn_exp2f(M - mx), w = __builtin_amdgcn_exp2f(m - mx);
    float ls = w * l;
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) ls += __shfl_xor(ls, o);
    sum = sum * a + ls;
    acc *= a;
    M = mx;
    for (int i0 = 0; i0 < n; i0 += G) {
      f4 v[G];
#pragma unroll
      for (int i = 0; i < G; ++i)
        v[i] = *reinterpret_cast<const f4 *>(sl + (size_t)(s0 + min(i0 + i, n - 1)) * block_rows * R);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const float wi = i0 + i < n ? __shfl(w, i0 + i) : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(wi, v[i][e], acc[e]);
      }
    }
  }
  const float inv = __fdiv_rn(1.0f, sum);
  if (col >= R) return;
  *reinterpret_cast<uint2 *>(O + (size_t)(mg.row0 + r) * R + col) =
      make_uint2(f2bf(acc[0] * inv) | ((uint32_t)f2bf(acc[1] * inv) << 16),
                 f2bf(acc[2] * inv) | ((uint32_t)f2bf(acc[3] * inv) << 16));
}

bool latent_rank_supported(int rank) {
  const int rc = rank / 64;
  return rank % 64 == 0 && (rc == 1 || rc == 2 || rc == 3 || rc == 4 || rc == 6 || rc == 8);
}

hipError_t launch_latent_attention(const char *blob, const PagedLists &pl, const uint16_t *q,
                                   const uint16_t *cache, uint16_t *o, float *slabs, float *ml,
                                   int rank, float scale, hipStream_t s) {
  if (pl.num_blocks <= 0) return hipSuccess;
  const float sl = scale * 1.4426950408889634f;
#define FFMI_LA2(RC, RT)                                                                        \
  hipLaunchKernelGGL((latent_attn_kernel<RC, RT>), dim3(pl.num_blocks), dim3(512), 0, s, blob,  \
                     pl.off_blocks, q, cache, o, slabs, ml, pl.heads, sl)
#define FFMI_LA(RC)                                                                             \
  case RC:                                                                                      \
    if (pl.row_tiles == 1) FFMI_LA2(RC, 1);                                                     \
    else if (pl.row_tiles == 2) FFMI_LA2(RC, 2);                                                \
    else if (pl.row_tiles == 4)                                                                 \
      hipLaunchKernelGGL((latent_attn_wide_kernel<RC>), dim3(std::min(pl.num_blocks, 256 * kLatentWide<RC>)), dim3(512), 0, s, \
                         blob, pl.off_blocks, pl.num_blocks, q, cache, o, slabs, ml, pl.heads, sl); \
    else return hipErrorInvalidValue;                                                           \
    if (pl.num_merges > 0)                                                                      \
      hipLaunchKernelGGL((latent_merge_kernel<RC>), dim3(pl.num_merges, pl.row_tiles * 16),     \
                         dim3(kMergeThreads<RC>), 0, s, blob, pl.off_merges, slabs, ml, o,                \
                         pl.row_tiles * 16);                                                    \
    break
  if (rank % 64) return hipErrorInvalidValue;
  switch (rank / 64) {
    FFMI_LA(1);
    FFMI_LA(2);
    FFMI_LA(3);
    FFMI_LA(4);
    FFMI_LA(6);
    FFMI_LA(8);
    default: return hipErrorInvalidValue;
  }
#undef FFMI_LA
#undef FFMI_LA2
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// attention, one workgroup per row (fp32, and bf16 ranks without an MFMA form)
// ---------------------------------------------------------------------------
constexpr int kRowsMaxRank = 2048;
template <class E>
__global__ __launch_bounds__(256) void latent_rows_kernel(const char *__restrict__ blob,
                                                          int off_blocks, const E *__restrict__ Q,
                                                          const E *__restrict__ cache,
                                                          E *__restrict__ O, int heads, int rank,
                                                          float scale) {
  __shared__ float sq[kRowsMaxRank], sp[256], red[4];
  __shared__ int srow[256];
  const PagedBlock bk = reinterpret_cast<const PagedBlock *>(blob + off_blocks)[blockIdx.x];
  const int r = blockIdx.y, tid = threadIdx.x;
  if (r >= bk.nrows) return;
  const int32_t *table = reinterpret_cast<const int32_t *>(blob) + bk.table;
  const size_t row = (size_t)bk.row0 + r;
  const int n = bk.pos0 + (int)(row - bk.seg_row) / heads + 1;  // visible positions
  for (int i = tid; i < rank; i += 256) sq[i] = ld_elem(Q + row * rank + i);
  float acc[kRowsMaxRank / 256];
#pragma unroll
  for (int i = 0; i < kRowsMaxRank / 256; ++i) acc[i] = 0.f;
  float m = -1e30f, l = 0.f;
  for (int j0 = 0; j0 < n; j0 += 256) {
    __syncthreads();
    const int j = j0 + tid;
    float sv = -INFINITY;
    if (j < n) {
      const int cr = table[j >> 6] * kPageTokens + (j & 63);
      srow[tid] = cr;
      const E *c = cache + (size_t)cr * rank;
      float a = 0.f;
      for (int i = 0; i < rank; ++i) a = fmaf(sq[i], ld_elem(c + i), a);
      sv = a * scale;
    }
    float mx = sv;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    const float mn = fmaxf(m, fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
    const float p = j < n ? expf(sv - mn) : 0.f;
    sp[tid] = p;
    float sum = p;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = sum;
    __syncthreads();
    const float al = expf(m - mn);
    l = l * al + (red[0] + red[1] + red[2] + red[3]);
    m = mn;
    const int cnt = min(256, n - j0);
#pragma unroll
    for (int i = 0; i < kRowsMaxRank / 256; ++i) {
      const int d = tid + i * 256;
      if (d >= rank) break;
      float a = acc[i] * al;
      for (int k = 0; k < cnt; ++k) a = fmaf(sp[k], ld_elem(cache + (size_t)srow[k] * rank + d), a);
      acc[i] = a;
    }
  }
  const float inv = __fdiv_rn(1.0f, l);
#pragma unroll
  for (int i = 0; i < kRowsMaxRank / 256; ++i) {
    const int d = tid + i * 256;
    if (d < rank) st_elem(O + row * rank + d, acc[i] * inv);
  }
}

hipError_t launch_latent_attention_rows(const char *blob, const PagedLists &pl, const void *q,
                                        const void *cache, void *o, int rank, float scale,
                                        bool bf16, hipStream_t s) {
  if (pl.num_blocks <= 0) return hipSuccess;
  if (rank > kRowsMaxRank || pl.num_merges > 0) return hipErrorInvalidValue;
  const dim3 grid(pl.num_blocks, pl.row_tiles * 16);
  if (bf16)
    hipLaunchKernelGGL(latent_rows_kernel<uint16_t>, grid, dim3(256), 0, s, blob, pl.off_blocks,
                       (const uint16_t *)q, (const uint16_t *)cache, (uint16_t *)o, pl.heads, rank,
                       scale);
  else
    hipLaunchKernelGGL(latent_rows_kernel<float>, grid, dim3(256), 0, s, blob, pl.off_blocks,
                       (const float *)q, (const float *)cache, (float *)o, pl.heads, rank, scale);
  return hipGetLastError();
}

}  // namespace ffmi
