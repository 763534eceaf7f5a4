// f32.hip -- the full-precision path: the reference's --use-full-precision
// (inference/spec_infer/spec_infer.cc:102, incr_decoding.cc:77), i.e. every
// operator of the LLaMA graph on DT_FLOAT -- weights, activations, KV cache,
// softmax.  The same operators as the half path (gemm.hip, attention.hip,
// norm.hip), restated for fp32 operands:
//  * Linear on v_mfma_f32_16x16x4_f32 -- exact fp32: the result is a k-ordered
//    fmaf chain per (wave, k range), no reduced-precision inputs (gfx950 has
//    no xf32), k ranges of a workgroup summed in a fixed order, the operands
//    through LDS rings of each wave's own;
//  * RMSNorm / ResidualRMSNorm with the sum of squares in fp64 (as the oracle,
//    then rounded once to fp32), fp32 residual adds;
//  * attention: one workgroup per (token, head) over the token's visible keys
//    (its prefix + its tree bits, the packed rule of attention.hip), fp32
//    scores, __expf-free softmax (expf), fp64 sum, 1/(sum + 1e-6)
//    (inc_multihead_self_attention.cu:532-547 on DT_FLOAT);
//  * softmax + argmax / arg-top-k on fp32 probabilities (softmax.cu:262-288,
//    argmax.cu:62-100, arg_topk.cu:339-448): lowest index among equal maxima.
// KV cache fp32, K[req][head][slot][d] and V[req][head][slot][d].
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "../ffmi_internal.h"

namespace ffmi {

// ---------------------------------------------------------------------------
// Linear: Y[T][N] = X[T][K] . W[N][K]^T (linear_kernels.cu:450-582, DT_FLOAT)
// ---------------------------------------------------------------------------
// (a * sigmoid(a)) * b
__device__ __forceinline__ float f32_silu_mul(float a, float b) {
  const float sg = __fdiv_rn(1.0f, __fadd_rn(1.0f, expf(-a)));
  return __fmul_rn(__fmul_rn(a, sg), b);
}

// The column block that workgroup b of n takes of a packed weight.  Workgroups go round the
// eight XCDs, so in their own order an XCD reads 2 KiB (8 columns: 1 KiB) of each 16 (8) of
// a band, always the same ones where the bands are of a round number of them: a part of its
// L2's channels.  There an XCD takes an eighth of the columns in one piece.  Rows / blocks in their
// own order / so, us: T = 4, 4096 x 2048 8.3 / 10.1 / 8.5, x 3072 11.3 / 12.9 / 10.7, x 4096 16.1 / 16.8 /
// 14.2, x 8192 30.3 / 27.8 / 23.1; 6144 x 2048 12.1 / 12.8 / 11.8; 12288 x 2048 18.9 / 19.9 / 18.7; gate/up 2 x
// 2048 x 4096 9.8 / 8.9 (blocks); T = 24, 4096 x 2048 10.1 / 11.6 / 10.5.  Other numbers of workgroups
// gain nothing by it or lose (32000 x 2048 46.2 -> 47.9, 11264 x 2048 18.1 -> 18.4; fewer than 256,
// 1024 x 3072 at T = 16 9.1 -> 9.4).
__device__ __forceinline__ int f32_column_block(int b, int n) {
  return n % 128 == 0 && n >= 256 ? (b & 7) * (n >> 3) + (b >> 3) : b;
}

// k quarters summed in wave order: 0 + 1 + 2 + 3 (fixed, deterministic), and stored
template <int MT, int NT>
__device__ __forceinline__ void f32_gemm_store(f4 (&acc)[MT][NT], f4 (*red)[MT * NT][64],
                                               float *__restrict__ Y, int T, int N, int row0, int col0,
                                               int wave, int lane) {
  if (wave > 0)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) red[wave - 1][m * NT + n][lane] = acc[m][n];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] += red[s][m * NT + n][lane];
  // C/D map: col = lane & 15, row = 4 * (lane >> 4) + i
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int col = col0 + n * 16 + (lane & 15);
      if (col >= N) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + m * 16 + 4 * (lane >> 4) + i;
        if (row < T) Y[(size_t)row * N + col] = acc[m][n][i];
      }
    }
}

// Four waves, each a quarter of the k-blocks of 32 and all MT x NT tiles of 16 x 16
// of the workgroup; the quarters are summed through LDS in wave order.  Operand map
// of v_mfma_f32_16x16x4_f32: lane l supplies A[row l&15][k l>>4] and B[k l>>4][col
// l&15]; the lane holds 16 B of X / W at k0 + 4*(l>>4) (+16), and MFMA j of a 16-k
// half takes element j: the four lane groups cover k0 + 4g + j, g = 0..3 -- all 16 k
// of the half.
// Neighbouring lanes of an operand want different rows, which the L1 serves one
// 16-byte access after another: read straight into registers (f32_gemm_kernel)
// that, not HBM or the MFMA, was the bound.  Here each wave copies its k-blocks to
// an LDS ring of its own, PF of them on their way, a row's 128 bytes to 8 lanes (its
// 16-byte pieces exchanged by the row's number: the operand reads then hit different
// banks), and reads the next block's operands while it multiplies this one's.
// Nothing is shared before the sum, so there is no barrier.  Blocks in turn use two sets
// of registers: moving a set (up to 64 registers a block, on the one wave of a SIMD that
// also issues the MFMAs) took 3-12% of a product (packed, us: T = 201, 2 x 4 tiles, N = 11264
// 108.6 -> 104.6, K = 5632 x N = 2048 53.9 -> 51.0; T = 75, 2 x 2, K = 5632 32.3 -> 28.9; T = 1000,
// 4 x 4, N = 11264 419 -> 406; T = 24, N = 32000, the stream of weights, 51.0 and 52.0).
template <int MT, int NT, int PF, bool PACKED = false>
__global__ __launch_bounds__(256) void f32_gemm_lds_kernel(const float *__restrict__ X,
                                                          const float *__restrict__ W,
                                                          float *__restrict__ Y, int T, int N, int K) {
  constexpr int F = MT + NT, PW = 2 * F;  // tiles of a k-block, its copies
  static_assert(PF * PW <= 63, "vmcnt");
  __shared__ f4 lds[4][PF][F][128];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = blockIdx.y * MT * 16, col0 = (PACKED ? f32_column_block(blockIdx.x, gridDim.x) : (int)blockIdx.x) * NT * 16;
  const int r = lane & 15, g = lane >> 4;
  const int nb = K >> 5;  // k-blocks of 32 (host-checked K % 32 == 0)
  const int kb0 = wave * nb / 4, n = (wave + 1) * nb / 4 - kb0;
  const int tiles = (N + 7) >> 3;  // PACKED: of 8 columns
  const float *src[PW];
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int f = p >> 1, row = 8 * (p & 1) + (lane >> 3), piece = (lane ^ row) & 7;
    if (f < MT) src[p] = X + (size_t)min(row0 + f * 16 + row, T - 1) * K + (size_t)kb0 * 32;
    else if (!PACKED) src[p] = W + (size_t)min(col0 + (f - MT) * 16 + row, N - 1) * K + (size_t)kb0 * 32;
    else src[p] = W + ((size_t)kb0 * tiles + min(((col0 >> 3) + 2 * (f - MT) + (p & 1)), tiles - 1)) * 256 + (lane >> 3) * 32;
    src[p] += piece * 4;
  }
  auto copy = [&](int kb, int slot) {
#pragma unroll
    for (int p = 0; p < PW; ++p)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void *)(src[p] + (size_t)kb * (PACKED && p >= 2 * MT ? tiles * 256 : 32)),
          (__attribute__((address_space(3))) void *)&lds[wave][slot][p >> 1][64 * (p & 1)], 16, 0, 0);
  };
  f4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = f4{0.f, 0.f, 0.f, 0.f};
  f4 va[F][2], vb[F][2];
  auto read = [&](int slot, f4 (&v)[F][2]) {
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int h = 0; h < 2; ++h) v[f][h] = lds[wave][slot][f][r * 8 + ((4 * h + g) ^ (r & 7))];
  };
  // s_waitcnt vmcnt(V) alone
  auto wait = [](auto V) { __builtin_amdgcn_s_waitcnt((V.value & 15) | 0x0f70 | ((V.value >> 4) << 14)); };
#pragma unroll
  for (int i = 0; i < PF; ++i)
    if (i < n) copy(i, i);
  if (n >= PF) wait(std::integral_constant<int, (PF - 1) * PW>{});
  else wait(std::integral_constant<int, 0>{});
  asm volatile("" ::: "memory");
  if (n > 0) read(0, va);
  int slot = 0;
  auto step = [&](int kb, f4 (&cur)[F][2], f4 (&nxt)[F][2]) {
    const int next = slot + 1 == PF ? 0 : slot + 1;
    // this block's operands are in registers; its slot takes block kb + PF
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    if (kb + PF < n) {
      copy(kb + PF, slot);
      wait(std::integral_constant<int, (PF - 1) * PW>{});
    } else {
      wait(std::integral_constant<int, 0>{});
    }
    asm volatile("" ::: "memory");
    if (kb + 1 < n) read(next, nxt);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int i = 0; i < NT; ++i)
            acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[m][h][j], cur[MT + i][h][j], acc[m][i], 0, 0, 0);
    slot = next;
  };
  int kb = 0;
  for (; kb + 1 < n; kb += 2) {
    step(kb, va, vb);
    step(kb + 1, vb, va);
  }
  if (kb < n) step(kb, va, vb);
  __syncthreads();
  auto red = reinterpret_cast<f4(*)[MT * NT][64]>(&lds[0][0][0][0]);
  static_assert(sizeof(lds) >= 3 * MT * NT * 64 * sizeof(f4), "sum buffer");
  f32_gemm_store<MT, NT>(acc, red, Y, T, N, row0, col0, wave, lane);
}

// Up to 16 rows (decoding) of packed weights (launch_pack_f32_blocks), where their stream
// is the time: one tile of 16 x 16, of which only what is needed is copied.  What a CU takes in comes back from its L1 in
// order, so that rows of X, from the L2, wait behind weights from HBM and take the place
// of weights in flight: in half tiles of columns, where they are two copies of three, XH
// (up to 8 rows) leaves out the other 8; whole tiles and pairs take the same time
// with and without (T = 8: 6144 x 2048 12.6 and 12.5 us, 12288 x 4096 35.0 and 35.1, gate/up 2 x 5632 x
// 2048 19.0 and 18.5, 2 x 11008 x 4096 64.3 and 65.1).  COLS = 8: half a tile of
// columns (the MFMA multiplies the other half for nothing), for widths whose 16-column
// workgroups leave CUs idle or unevenly loaded.  PAIR: columns 0..7 of the tile are
// gate's, 8..15 up's (W: F rows of gate, then F of up), and silu(gate) up goes out
// (f32_silu_mul_kernel's arithmetic).  The sums are the other forms', in their order.
template <int PF, bool XH, int COLS, bool PAIR>
__global__ __launch_bounds__(256) void f32_gemm_few_kernel(const float *__restrict__ X, const float *__restrict__ Wp,
                                                          float *__restrict__ Y, int T, int N, int K) {
  static_assert(COLS == 16 || COLS == 8, "columns of a workgroup");
  static_assert(!PAIR || COLS == 8, "a tile of gate and up columns");
  constexpr int CX = XH ? 1 : 2, CW = COLS == 8 && !PAIR ? 1 : 2, PW = CX + CW;  // copies of 8 rows
  static_assert(PF * PW <= 63, "vmcnt");
  __shared__ f4 lds[4][PF][PW][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col0 = f32_column_block(blockIdx.x, gridDim.x) * COLS, r = lane & 15, g = lane >> 4;
  const int nb = K >> 5;  // k-blocks of 32 (host-checked K % 32 == 0)
  const int kb0 = wave * nb / 4, n = (wave + 1) * nb / 4 - kb0;
  const int tiles = ((PAIR ? 2 * N : N) + 7) >> 3;  // of 8 columns: a k-block of W
  const float *src[PW];
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int row = lane >> 3, piece = (lane ^ row) & 7, c = p - CX;
    if (c < 0) src[p] = X + (size_t)min(8 * p + row, T - 1) * K + (size_t)kb0 * 32;
    else src[p] = Wp + ((size_t)kb0 * tiles + (PAIR ? c * (N >> 3) + (col0 >> 3) : min((col0 >> 3) + c, tiles - 1))) * 256 + row * 32;
    src[p] += piece * 4;
  }
  auto copy = [&](int kb, int slot) {
#pragma unroll
    for (int p = 0; p < PW; ++p)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void *)(src[p] + (size_t)kb * (p < CX ? 32 : tiles * 256)),
          (__attribute__((address_space(3))) void *)&lds[wave][slot][p][0], 16, 0, 0);
  };
  f4 acc[1][1] = {{f4{0.f, 0.f, 0.f, 0.f}}};
  f4 va[2][2], vb[2][2];  // [X, W][half of the k-block], of blocks in turn
  // (rows that were not copied: the first 8 again, in rows and columns that nobody takes)
  const int rx = XH ? 0 : r >> 3, rw = CX + (CW == 1 ? 0 : r >> 3);
  auto read = [&](int slot, f4 (&v)[2][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = (r & 7) * 8 + ((4 * h + g) ^ (r & 7));
      v[0][h] = lds[wave][slot][rx][at];
      v[1][h] = lds[wave][slot][rw][at];
    }
  };
  auto wait = [](auto V) {  // vmcnt(V) alone
    __builtin_amdgcn_s_waitcnt((V.value & 15) | 0x0f70 | ((V.value >> 4) << 14));
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int i = 0; i < PF; ++i)
    if (i < n) copy(i, i);
  if (n >= PF) wait(std::integral_constant<int, (PF - 1) * PW>{});
  else wait(std::integral_constant<int, 0>{});
  if (n > 0) read(0, va);
  int slot = 0;
  // Block kb.  Its eight products are one chain (the sums' order), 32 cycles each, which is the
  // time where few columns leave a wave alone on its SIMD: copies, waits and reads go into the
  // gaps between them, and blocks in turn use two sets of registers (moved from one set to
  // the other, and everything before the first product: K 5632 x N 2048 13.3 us at T = 4, so 10.9, 0.12 us
  // a block of which the chain is all; 2048 x 2048 6.6 and 5.5, 6144 x 2048 11.6 and 10.9).
  // MORE: block kb + PF exists; V: copies that may be out when block kb + 1 is read.
  auto step = [&](auto MORE, auto V, int kb, const f4 (&cur)[2][2], f4 (&nxt)[2][2]) {
    const int next = slot + 1 == PF ? 0 : slot + 1;
    const auto mul = [&](int h, int j) {
      __builtin_amdgcn_sched_barrier(0);
      acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[0][h][j], cur[1][h][j], acc[0][0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this block's operands are in registers
    asm volatile("" ::: "memory");
    mul(0, 0);
    if constexpr (MORE.value) copy(kb + PF, slot);
    mul(0, 1);
    wait(V);
    read(next, nxt);  // (behind the last block: a slot that nobody needs)
    mul(0, 2), mul(0, 3);
    mul(1, 0), mul(1, 1), mul(1, 2), mul(1, 3);
    slot = next;
  };
  const std::true_type yes{};
  const std::integral_constant<int, (PF - 1) * PW> all{};
  int kb = 0;
  for (; kb + 1 + PF < n; kb += 2) {
    step(yes, all, kb, va, vb);
    step(yes, all, kb + 1, vb, va);
  }
  const auto turn = [&] {
#pragma unroll
    for (int f = 0; f < 2; ++f) va[f][0] = vb[f][0], va[f][1] = vb[f][1];
  };
  if (kb + PF < n) {
    step(yes, all, kb++, va, vb);
    turn();
  }
  // the last PF blocks, without copies
  const auto drain = [&](auto REM) {
    if (n - kb != REM.value) return;
    step(std::false_type{}, std::integral_constant<int, (REM.value > 2 ? REM.value - 2 : 0) * PW>{}, kb++, va, vb);
    turn();
  };
  const auto drains = [&](const auto &self, auto REM) -> void {
    drain(REM);
    if constexpr (REM.value > 1) self(self, std::integral_constant<int, REM.value - 1>{});
  };
  drains(drains, std::integral_constant<int, PF>{});
  __syncthreads();
  auto red = reinterpret_cast<f4(*)[1][64]>(&lds[0][0][0][0]);
  static_assert(sizeof(lds) >= 3 * 64 * sizeof(f4), "sum buffer");
  if constexpr (COLS == 16) {
    f32_gemm_store<1, 1>(acc, red, Y, T, N, 0, col0, wave, lane);
  } else {
    if (wave > 0) red[wave - 1][0][lane] = acc[0][0];
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int s = 0; s < 3; ++s) acc[0][0] += red[s][0][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = acc[0][0][i];
      if constexpr (PAIR) v = f32_silu_mul(v, __shfl_xor(v, 8));  // (lanes of columns 0..7 hold gate's)
      const int row = 4 * g + i, col = col0 + r;
      if (r < 8 && col < N && row < T) Y[(size_t)row * N + col] = v;
    }
  }
}

// The same sums from operands read straight into registers, for rows that are not of
// 16-byte pieces (the copies to LDS are 16 bytes each).
template <int MT, int NT>
__global__ __launch_bounds__(256) void f32_gemm_kernel(const float *__restrict__ X,
                                                      const float *__restrict__ W,
                                                      float *__restrict__ Y, int T, int N, int K) {
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6;
  const int row0 = blockIdx.y * MT * 16, col0 = blockIdx.x * NT * 16;
  const int r = lane & 15, g = lane >> 4;
  const int nb = K >> 5;  // k-blocks of 32 (host-checked K % 32 == 0)
  const int kb0 = ks * nb / 4, kb1 = (ks + 1) * nb / 4;
  const float *xp[MT], *wp[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = X + (size_t)min(row0 + m * 16 + r, T - 1) * K + 4 * g;
#pragma unroll
  for (int n = 0; n < NT; ++n) wp[n] = W + (size_t)min(col0 + n * 16 + r, N - 1) * K + 4 * g;
  __shared__ f4 red[3][MT * NT][64];
  f4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
  f4 a[2][MT][2], b[2][NT][2];  // double-buffered k-block operands
  auto load = [&](int buf, int kb) {
    const int k = kb * 32;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      a[buf][m][0] = *reinterpret_cast<const f4 *>(xp[m] + k);
      a[buf][m][1] = *reinterpret_cast<const f4 *>(xp[m] + k + 16);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      b[buf][n][0] = *reinterpret_cast<const f4 *>(wp[n] + k);
      b[buf][n][1] = *reinterpret_cast<const f4 *>(wp[n] + k + 16);
    }
  };
  auto mma = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[buf][m][h][j], b[buf][n][h][j],
                                                             acc[m][n], 0, 0, 0);
  };
  if (kb0 < kb1) {
    load(0, kb0);
    int kb = kb0;
    for (; kb + 2 <= kb1; kb += 2) {  // next block in flight while this one multiplies
      load(1, kb + 1);
      mma(0);
      if (kb + 2 < kb1) load(0, kb + 2);
      mma(1);
    }
    if (kb < kb1) mma(0);
  }
  f32_gemm_store<MT, NT>(acc, red, Y, T, N, row0, col0, ks, lane);
}

// Forms of more than 16 rows: the one with the least work on the busiest CU, workgroups
// of a CU in rounds of 256 times a workgroup's tiles, times what a tile costs in that
// form next to a 4 x 4 one (measured at N 2048-32000, K 2048 and 4096, T 24-1024; 2.3 us
// a tile at K = 2048).  All forms add up an output in the same order.  T = 201, K = 2048:
// N = 2048 2 x 4 tiles 21.4 us, 4 x 4 37.1 (41.2 from registers); N = 11264 105 and
// 112 (123); N = 32000 298 and 306 (329).  Two 2 x 2 workgroups share a CU, and the third
// round of three shares with none: it counts 1.3 (N = 6144, T = 120 43.3 us, 4 x 4 39.7; of 120
// products 6 change form by it, 5 to a faster one: 0.2% above the fastest form on average,
// 0.5% without).
template <bool PACKED>
static void f32_gemm_many(const float *X, const float *W, float *Y, int T, int N, int K, hipStream_t s) {
  const auto tiles = [&](int mt, int nt) {
    return dim3((N + 16 * nt - 1) / (16 * nt), (T + 16 * mt - 1) / (16 * mt));
  };
  struct Form {
    int mt, nt;
    double cost;
  };
  static const Form forms[] = {{4, 4, 1.0}, {3, 4, 1.04}, {2, 4, 1.11}, {3, 2, 1.22}, {2, 2, 1.24}, {2, 1, 1.5}};
  int best = 0;
  double least = 1e30;
  for (int i = 0; i < 6; ++i) {
    const dim3 g = tiles(forms[i].mt, forms[i].nt);
    const size_t rounds = ((size_t)g.x * g.y + 255) / 256;
    const double c = (rounds == 3 && forms[i].mt * forms[i].nt == 4 ? 3.3 : (double)rounds) * forms[i].mt * forms[i].nt * forms[i].cost;
    if (c < least) least = c, best = i;
  }
#define FFMI_F32_GEMM(MT, NT, PF)                                                                           \
  hipLaunchKernelGGL((f32_gemm_lds_kernel<MT, NT, PF, PACKED>), tiles(MT, NT), dim3(256), 0, s, X, W, Y, T, \
                     N, K)
  if (best == 0) FFMI_F32_GEMM(4, 4, 2);
  else if (best == 1) FFMI_F32_GEMM(3, 4, 2);
  else if (best == 2) FFMI_F32_GEMM(2, 4, 2);
  else if (best == 3) FFMI_F32_GEMM(3, 2, 2);
  else if (best == 4) FFMI_F32_GEMM(2, 2, 2);
  else FFMI_F32_GEMM(2, 1, 3);
#undef FFMI_F32_GEMM
}

hipError_t launch_gemm_f32(const float *X, const float *W, float *Y, int T, int N, int K,
                           hipStream_t s) {
  if (T <= 0 || N <= 0) return hipSuccess;
  if (K <= 0 || K % 32) return hipErrorInvalidValue;
  const dim3 one((N + 15) / 16, (T + 15) / 16), four((N + 63) / 64, (T + 63) / 64), block(256);
  if (((uintptr_t)X | (uintptr_t)W) & 15) {
    if (T <= 16) hipLaunchKernelGGL((f32_gemm_kernel<1, 1>), one, block, 0, s, X, W, Y, T, N, K);
    else hipLaunchKernelGGL((f32_gemm_kernel<4, 4>), four, block, 0, s, X, W, Y, T, N, K);
    return hipGetLastError();
  }
  // Up to 16 rows: a ring of four k-blocks (N = 2048, K = 5632: 13.9 us, 22.7 from registers)
  // takes 64 KiB, two workgroups to a CU, which is too few where each has little to
  // read: of two for short K (N = 32000, T = 8: K = 512 14.3 us, 18.1 with four, 16.0 from
  // registers; K = 2048, T = 1 48.2 and 46.1), and up to 4 rows, which fall into one access
  // of a load, registers for the shortest (N = 32000, K = 256, T = 1: 7.6, ring of two 8.8,
  // of four 11.7; T = 16 10.4, 9.5 and 12.6).
  if (T <= 4 && K <= 256)
    hipLaunchKernelGGL((f32_gemm_kernel<1, 1>), one, block, 0, s, X, W, Y, T, N, K);
  else if (T <= 16 && (K <= 512 || (K <= 1024 && N >= 4096)))
    hipLaunchKernelGGL((f32_gemm_lds_kernel<1, 1, 2>), one, block, 0, s, X, W, Y, T, N, K);
  else if (T <= 16)
    hipLaunchKernelGGL((f32_gemm_lds_kernel<1, 1, 4>), one, block, 0, s, X, W, Y, T, N, K);
  else
    f32_gemm_many<false>(X, W, Y, T, N, K, s);
  return hipGetLastError();
}

// Short rows stay as they lie: their workgroups read a few KiB each, in one piece, which
// blocks scatter over as many bands.  T = 1, 4, 8 and 16, us, rows / blocks: N 32000 x K 256 7.4 / 9.7,
// 8.1 / 10.0, 8.8 / 10.1, 9.1 / 10.5; x 512 13.2 / 15.2, 13.5 / 15.5, 13.8 / 15.7, 14.4 / 16.4; x 768 19.7 / 20.3 .. 21.9 /
// 22.3; 2304 x 768 3.8 / 4.0 .. 4.1 / 4.3; 4096 x 1024 5.9 / 6.5 .. 6.2 / 6.7; equal above 16 rows.  From
// 1280 on blocks are 0.8 (4096 x 2048) to 1.4 times as fast (K 11008 x N 4096), 1.0 to 1.2 from 5120
// columns on; a model's steps of 1, 4 and 12 tokens are 2, 2 and 2% faster with this line at width 256,
// 2% at 512, 3% at 768, 1% at 1024.  Gate and up are in blocks whatever K is: 1.1 to 1.5 times as fast as
// rows and a unit of their own.
bool f32_in_blocks(int K) { return K >= 1280; }

// Packed weights (launch_pack_f32_blocks).  Up to 16 rows, T = 4, us, rows as they lie and
// packed: 12288 x 4096 43.0 -> 34.4, 22016 x 4096 72.3 -> 62.7, K 11008 x N 4096 46.0 -> 29.3,
// 4096 x 4096 17.6 -> 13.4, 6144 x 2048 12.4 -> 10.9, 11264 x 2048 19.3 -> 18.1, K 5632 x N 2048
// 14.2 -> 10.2, 2048 x 2048 7.0 -> 5.5.
//  * Half tiles of columns where whole ones are at most half as many as CUs; at 256 and above
//    they lose (4096 x 4096 13.4 -> 14.7, K 11008 x N 4096 29.3 -> 33.1).  A workgroup is then alone
//    on its CU: a ring of six k-blocks (K 5632 x N 2048 10.9 -> 10.2, 768 x 3072 6.7 -> 6.5; above 8
//    rows, which copy more of X, of four: 12.6 and 12.7).
//  * A ring of two k-blocks, four workgroups to a CU, where there are several rounds of
//    them and K is short (6144 x 2048 11.4 -> 10.9, 32000 x 4096 96.1 -> 91.1; but 4096 x
//    4096, one round, 13.4 and 14.9, and K 11008 29.3 and 34.6).
static bool short_ring(int workgroups, int K) { return workgroups > 256 && K <= 4096; }
hipError_t launch_gemm_f32_packed(const float *X, const float *Wp, float *Y, int T, int N, int K, hipStream_t s) {
  if (T <= 0 || N <= 0) return hipSuccess;
  if (K <= 0 || K % 32 || (((uintptr_t)X | (uintptr_t)Wp) & 15)) return hipErrorInvalidValue;
  const int wgs = (N + 15) / 16;
  if (T > 16) f32_gemm_many<true>(X, Wp, Y, T, N, K, s);
  else if (wgs <= 128 && T <= 8)
    hipLaunchKernelGGL((f32_gemm_few_kernel<6, true, 8, false>), dim3((N + 7) / 8), dim3(256), 0, s, X, Wp, Y, T, N, K);
  else if (wgs <= 128)
    hipLaunchKernelGGL((f32_gemm_few_kernel<4, false, 8, false>), dim3((N + 7) / 8), dim3(256), 0, s, X, Wp, Y, T, N, K);
  else if (short_ring(wgs, K))
    hipLaunchKernelGGL((f32_gemm_few_kernel<2, false, 16, false>), dim3(wgs), dim3(256), 0, s, X, Wp, Y, T, N, K);
  else
    hipLaunchKernelGGL((f32_gemm_few_kernel<4, false, 16, false>), dim3(wgs), dim3(256), 0, s, X, Wp, Y, T, N, K);
  return hipGetLastError();
}

// out [T][F] = silu(X Wg^T) * (X Wu^T), Wp: the F rows of gate, then up's, packed; gu: room
// for [T][2 F] (more than 16 rows take the product and its unit one after the other).
// Rings of two and of four k-blocks, T = 4: 2 x 3072 x 768 6.1 and 6.3 us, 2 x 5632 x 2048 18.4 and
// 18.1 (T = 1 18.1 and 17.2), 2 x 11008 x 4096 63.7 and 62.7.
hipError_t launch_gate_up_f32_packed(const float *X, const float *Wp, float *gu, float *out, int T, int F, int K,
                                     hipStream_t s) {
  if (T <= 0 || F <= 0) return hipSuccess;
  if (T > 16 || F % 8) {
    const hipError_t e = launch_gemm_f32_packed(X, Wp, gu, T, 2 * F, K, s);
    return e != hipSuccess ? e : launch_silu_mul_f32(gu, gu + F, out, T, F, 2 * (size_t)F, 2 * (size_t)F, s);
  }
  if (K <= 0 || K % 32 || (((uintptr_t)X | (uintptr_t)Wp) & 15)) return hipErrorInvalidValue;
  if (F / 8 > 256 && K < 2048)
    hipLaunchKernelGGL((f32_gemm_few_kernel<2, false, 8, true>), dim3(F / 8), dim3(256), 0, s, X, Wp, out, T, F, K);
  else
    hipLaunchKernelGGL((f32_gemm_few_kernel<4, false, 8, true>), dim3(F / 8), dim3(256), 0, s, X, Wp, out, T, F, K);
  return hipGetLastError();
}

// Blocks of 8 columns x 32 k (1 KiB, one copy to LDS), k-block after k-block: column n's
// element k at ((k / 32 * tiles + n / 8) * 8 + n % 8) * 32 + k % 32, tiles = ceil(N / 8).
// Read k-block by k-block, the chip walks one band of memory instead of 128 bytes of each
// of thousands of rows.
__global__ __launch_bounds__(256) void pack_f32_blocks_kernel(const float *__restrict__ src, int ld, float *__restrict__ dst,
                                                            int tiles, int n0, int rows, int K) {
  const size_t pieces = (size_t)rows * (K >> 2);
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < pieces; i += (size_t)gridDim.x * 256) {
    const int row = (int)(i / (K >> 2)), k = (int)(i % (K >> 2)) * 4, n = n0 + row;
    const f4 v = *reinterpret_cast<const f4 *>(src + (size_t)row * ld + k);
    *reinterpret_cast<f4 *>(dst + (((size_t)(k >> 5) * tiles + (n >> 3)) * 8 + (n & 7)) * 32 + (k & 31)) = v;
  }
}

hipError_t launch_pack_f32_blocks(const float *src, int ld, float *dst, int N, int n0, int rows, int K, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  if (K <= 0 || K % 32 || ld % 4 || n0 < 0 || n0 + rows > N || (((uintptr_t)src | (uintptr_t)dst) & 15))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(pack_f32_blocks_kernel, dim3((unsigned)std::min<size_t>(((size_t)rows * (K / 4) + 255) / 256, 8192)),
                     dim3(256), 0, s, src, ld, dst, (N + 7) / 8, n0, rows, K);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// block reductions (256 threads)
// ---------------------------------------------------------------------------
template <class V, class Op>
__device__ __forceinline__ V block_reduce256(V v, V *sh, Op op) {
  // fixed order: lanes pairwise by xor within the wave, then waves 0..3
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off));
  const int w = threadIdx.x >> 6;
  __syncthreads();  // sh may still be read from the previous reduction
  if ((threadIdx.x & 63) == 0) sh[w] = v;
  __syncthreads();
  V t = sh[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) t = op(t, sh[i]);
  return t;
}

// ---------------------------------------------------------------------------
// RMSNorm / ResidualRMSNorm (rms_norm_kernels.cu:97-124,
// residual_rms_norm_kernels.cu:98-131) on fp32: r = x1 (+ x2); rms =
// 1/sqrt(sum(r^2)/H + eps) (sum in fp64, rounded once); out = (r * rms) * w.
// gather (layer 0): x1 is the embedding table, row t = the token's row
// (embedding_kernels.cu:233-244), res_out gets the looked-up row.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void f32_rmsnorm_kernel(
    const float *x1, const float *__restrict__ x2, const float *__restrict__ w, float *res_out,
    float *__restrict__ out, int H, float eps, const char *__restrict__ gather, const int32_t *__restrict__ rows) {
  __shared__ double sh[4];
  const int row = rows ? rows[blockIdx.x] : blockIdx.x;  // (rows: the output's row i is of input row rows[i])
  const float *a = gather ? x1 + (size_t)batch_view(gather).tokens[row].token_id * H
                          : x1 + (size_t)row * H;
  const float *b = x2 ? x2 + (size_t)row * H : nullptr;
  double ss = 0.0;
  for (int j = threadIdx.x; j < H; j += blockDim.x) {
    const float v = b ? __fadd_rn(a[j], b[j]) : a[j];
    if (res_out) res_out[(size_t)row * H + j] = v;
    ss += (double)v * (double)v;
  }
  ss = block_reduce256(ss, sh, [](double p, double q) { return p + q; });
  const float sum = (float)ss;
  // sqrtf: the correctly rounded square root (HIP's __fsqrt_rn is the native
  // v_sqrt_f32, ~1 ulp, unless OCML_BASIC_ROUNDED_OPERATIONS is defined)
  const float rms = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)H), eps)));
  // (res_out may alias x1: read back this thread's own sums, never x1 + x2 again)
  for (int j = threadIdx.x; j < H; j += blockDim.x) {
    const float v = res_out ? res_out[(size_t)row * H + j] : (b ? __fadd_rn(a[j], b[j]) : a[j]);
    out[(size_t)blockIdx.x * H + j] = __fmul_rn(__fmul_rn(v, rms), w[j]);
  }
}

// The same for rows of 16-byte pieces, NV of them per thread: the row is read once,
// 16 bytes per load and all loads in flight together, and stays in registers.  A row
// of 2048 (4 tokens, residual): 8.4 us an element at a time, 4.7 this way, which is
// three round trips to memory and the launch.
// FETCH: the rows that the step's tokens name (BlobFetch).  A token's id is one trip to
// the host's memory, on which the blob's copy goes along (a copy before, the header's
// offset and the id from device memory: 2.8 us of their own and two trips more here).
template <int NV, bool FETCH = false>
__global__ __launch_bounds__(256) void f32_rmsnorm_vec_kernel(
    const float *x1, const float *__restrict__ x2, const float *__restrict__ w, float *res_out,
    float *__restrict__ out, int H, float eps, std::conditional_t<FETCH, BlobFetch, const int32_t *> from) {
  __shared__ double sh[4];
  size_t row;
  const float *a;
  if constexpr (FETCH) {
    row = (size_t)blockIdx.x * H;
    a = x1 + (size_t)reinterpret_cast<const ffmi_token_info *>(from.host + from.off_tokens)[blockIdx.x].token_id * H;
    const uint4 *src = reinterpret_cast<const uint4 *>(from.host);
    const int n16 = (int)((from.bytes + 15) / 16);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n16; i += gridDim.x * 256)
      reinterpret_cast<uint4 *>(from.dev)[i] = src[i];
  } else {
    row = (size_t)(from ? from[blockIdx.x] : blockIdx.x) * H;
    a = x1 + row;
  }
  f4 v[NV], y[NV], g[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int j = min((int)(threadIdx.x + 256 * i) * 4, H - 4);
    v[i] = *reinterpret_cast<const f4 *>(a + j);
    if (x2) y[i] = *reinterpret_cast<const f4 *>(x2 + row + j);
    g[i] = *reinterpret_cast<const f4 *>(w + j);
  }
  double ss = 0.0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int j = (threadIdx.x + 256 * i) * 4;
    if (j >= H) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (x2) v[i][e] = __fadd_rn(v[i][e], y[i][e]);
      ss += (double)v[i][e] * (double)v[i][e];
    }
    if (res_out) *reinterpret_cast<f4 *>(res_out + row + j) = v[i];
  }
  ss = block_reduce256(ss, sh, [](double p, double q) { return p + q; });
  const float sum = (float)ss;
  const float rms = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)H), eps)));
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int j = (threadIdx.x + 256 * i) * 4;
    if (j >= H) continue;
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = __fmul_rn(__fmul_rn(v[i][e], rms), g[i][e]);
    *reinterpret_cast<f4 *>(out + (size_t)blockIdx.x * H + j) = o;
  }
}

// rows and buffers of 16-byte pieces, up to 8 per thread (more would spill)
static bool f32_rows_in_pieces(const float *x1, const float *x2, const float *w, const float *res_out,
                               const float *out, int H) {
  return H > 0 && H % 4 == 0 && H <= 8192 &&
         (((uintptr_t)x1 | (uintptr_t)x2 | (uintptr_t)w | (uintptr_t)res_out | (uintptr_t)out) & 15) == 0;
}
hipError_t launch_rmsnorm_f32(const float *x1, const float *x2, const float *w, float *res_out,
                              float *out, int T, int H, float eps, hipStream_t s, const int32_t *rows) {
  if (rows && res_out) return hipErrorInvalidValue;
  if (T <= 0) return hipSuccess;
#define FFMI_NORM(NV) \
  hipLaunchKernelGGL(f32_rmsnorm_vec_kernel<NV>, dim3(T), dim3(256), 0, s, x1, x2, w, res_out, out, H, eps, rows)
  if (!f32_rows_in_pieces(x1, x2, w, res_out, out, H))
    hipLaunchKernelGGL(f32_rmsnorm_kernel, dim3(T), dim3(256), 0, s, x1, x2, w, res_out, out, H, eps, nullptr, rows);
  else if (H <= 1024) FFMI_NORM(1);
  else if (H <= 2048) FFMI_NORM(2);
  else if (H <= 4096) FFMI_NORM(4);
  else FFMI_NORM(8);
#undef FFMI_NORM
  return hipGetLastError();
}
hipError_t launch_embed_rmsnorm_f32(const float *table, const BlobFetch &blob, const float *w, float *res_out,
                                    float *out, int T, int H, float eps, hipStream_t s) {
  if (!res_out || blob.off_tokens <= 0 || blob.bytes > (size_t)1 << 30 ||
      (((uintptr_t)blob.host | (uintptr_t)blob.dev) & 15))
    return hipErrorInvalidValue;
  if (T <= 0) return hipSuccess;
#define FFMI_NORM(NV)                                                                                                 \
  hipLaunchKernelGGL((f32_rmsnorm_vec_kernel<NV, true>), dim3(T), dim3(256), 0, s, table, nullptr, w, res_out, out, H, \
                     eps, blob)
  if (!f32_rows_in_pieces(table, nullptr, w, res_out, out, H)) {
    if (const hipError_t e = hipMemcpyAsync(blob.dev, blob.host, blob.bytes, hipMemcpyHostToDevice, s)) return e;
    hipLaunchKernelGGL(f32_rmsnorm_kernel, dim3(T), dim3(256), 0, s, table, nullptr, w, res_out, out, H, eps,
                       (const char *)blob.dev, nullptr);
  } else if (H <= 1024) FFMI_NORM(1);
  else if (H <= 2048) FFMI_NORM(2);
  else if (H <= 4096) FFMI_NORM(4);
  else FFMI_NORM(8);
#undef FFMI_NORM
  return hipGetLastError();
}

// SigmoidSiluMulti (sigmoid_silu_multi.cu:37-47) on fp32: out[t][f] =
// (a * sigmoid(a)) * b with a = A[t*lda + f], b = B[t*ldb + f] (the model's
// [T][2F] gate|up product: B = A + F, lda = ldb = 2F)
__global__ void f32_silu_mul_kernel(const float *__restrict__ A, const float *__restrict__ B,
                                    float *__restrict__ out, int T, int F, size_t lda,
                                    size_t ldb) {
  const size_t n = (size_t)T * F;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / F, f = i % F;
    const float a = A[t * lda + f], b = B[t * ldb + f];
    out[i] = f32_silu_mul(a, b);
  }
}

hipError_t launch_silu_mul_f32(const float *A, const float *B, float *out, int T, int F,
                               size_t lda, size_t ldb, hipStream_t s) {
  if (T <= 0 || F <= 0) return hipSuccess;
  const size_t n = (size_t)T * F;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(f32_silu_mul_kernel, dim3(blocks), dim3(256), 0, s, A, B, out, T, F, lda,
                     ldb);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// KV update: RoPE (apply_rotary_embedding_hf, inc...cu:664-738: pair
// (i, i + d/2), products rounded then summed) on q and k, K/V stored at the
// token's cache slot, and -- TREE -- the rotated k / v staged in row t for the
// next step's commits (tree_inc...cu:335-396 reads them).  Grid (T, heads),
// d/2 threads.
// ---------------------------------------------------------------------------
struct KvUpdateF32 {  // elements i and i + d / 2 of a (token, head)
  float q0, q1, k0, k1, va, vb;
};
__device__ __forceinline__ KvUpdateF32 f32_kv_update(const ffmi_token_info &tk, int t, int hd, int i,
                                                     const float *__restrict__ qkv, const float *__restrict__ rope,
                                                     int max_rope_pos, float *__restrict__ kc, float *__restrict__ vc,
                                                     float *__restrict__ stage, int heads, int d, int slots) {
  const int half = d / 2, Hl = heads * d;
  const float *row = qkv + (size_t)t * 3 * Hl + hd * d;
  const int p = min(max(tk.pos, 0), max_rope_pos - 1);
  const float c = rope[((size_t)p * half + i) * 2], sn = rope[((size_t)p * half + i) * 2 + 1];
  const float qa = row[i], qb = row[i + half];
  const float ka = row[Hl + i], kb = row[Hl + i + half];
  const float va = row[2 * Hl + i], vb = row[2 * Hl + i + half];
  const float q0 = __fsub_rn(__fmul_rn(qa, c), __fmul_rn(qb, sn));
  const float q1 = __fadd_rn(__fmul_rn(qa, sn), __fmul_rn(qb, c));
  const float k0 = __fsub_rn(__fmul_rn(ka, c), __fmul_rn(kb, sn));
  const float k1 = __fadd_rn(__fmul_rn(ka, sn), __fmul_rn(kb, c));
  if (tk.store_slot >= 0 && tk.store_slot < slots) {
    const size_t base = (((size_t)tk.req * heads + hd) * slots + tk.store_slot) * d;
    kc[base + i] = k0;
    kc[base + i + half] = k1;
    vc[base + i] = va;
    vc[base + i + half] = vb;
  }
  if (stage) {
    float *st = stage + (size_t)t * 2 * Hl + hd * d;
    st[i] = k0;
    st[i + half] = k1;
    st[Hl + i] = va;
    st[Hl + i + half] = vb;
  }
  return {q0, q1, k0, k1, va, vb};
}
__global__ void f32_kv_update_kernel(const char *__restrict__ blob, const float *__restrict__ qkv,
                                     const float *__restrict__ rope, int max_rope_pos,
                                     float *__restrict__ qbuf, float *__restrict__ kc,
                                     float *__restrict__ vc, float *__restrict__ stage, int heads,
                                     int d, int slots) {
  const int t = blockIdx.x, hd = blockIdx.y, i = threadIdx.x;
  if (i >= d / 2) return;
  const ffmi_token_info tk = batch_view(blob).tokens[t];
  const KvUpdateF32 u = f32_kv_update(tk, t, hd, i, qkv, rope, max_rope_pos, kc, vc, stage, heads, d, slots);
  float *qo = qbuf + (size_t)t * heads * d + hd * d;
  qo[i] = u.q0;
  qo[i + d / 2] = u.q1;
}

// commit_tokens_kernel (tree_inc...cu:335-396): accepted tokens of the
// previous verify batch move from their staging row to their depth slot
__global__ void f32_commit_kernel(const char *__restrict__ blob, const float *__restrict__ stage,
                                  float *__restrict__ kc, float *__restrict__ vc, int heads, int d,
                                  int slots) {
  const int ci = blockIdx.x, hd = blockIdx.y;
  const BatchView bv = batch_view(blob);
  const ffmi_commit_info cm = bv.commits[ci];
  if (cm.depth < 0 || cm.depth >= slots) return;
  const int Hl = heads * d;
  const float *st = stage + (size_t)cm.src_token * 2 * Hl + hd * d;
  const size_t base = (((size_t)cm.req * heads + hd) * slots + cm.depth) * d;
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    kc[base + i] = st[i];
    vc[base + i] = st[Hl + i];
  }
}

hipError_t launch_kv_update_f32(const char *blob, int T, int C, const float *qkv, const float *rope,
                                int max_rope_pos, float *qbuf, float *kc, float *vc,
                                float *stage, int heads, int d, int slots, hipStream_t s) {
  // commits first (the reference's commit-then-store order), from the rows
  // the previous step staged; this step's stores then overwrite the stage
  if (C > 0) {
    if (!stage) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f32_commit_kernel, dim3(C, heads), dim3(64), 0, s, blob, stage, kc, vc,
                       heads, d, slots);
  }
  if (T > 0)
    hipLaunchKernelGGL(f32_kv_update_kernel, dim3(T, heads), dim3(d / 2), 0, s, blob, qkv, rope,
                       max_rope_pos, qbuf, kc, vc, stage, heads, d, slots);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Attention of one (token, head): keys [0, prefix_len) plus the tree slots
// whose bit the token's visibility word holds (attention.hip key_visible);
// scores in LDS.  8 lanes share a key's dot product and D / 4 lanes a key's
// values, 16 bytes each, so that neighbouring lanes read whole lines, with four
// passes' loads in flight (a thread per key and a thread per output element, one
// load after another, took 23.9 us for 4 tokens x 16 heads, d = 128, about 160
// keys, now 6.5); output groups are summed in group order.
// UPDATE (a step of one token per request: no other workgroup's keys are this step's):
// the token's KV update first, its own key and value from LDS, the rest as it lies in the
// cache -- one launch of 7.8 us for two of 4.0 and 7.0 (4 tokens x 16 heads).
// ---------------------------------------------------------------------------
struct KvUpdateArgs {
  const float *qkv = nullptr, *rope = nullptr;
  int max_rope_pos = 0;
  float *kc = nullptr, *vc = nullptr, *stage = nullptr;
};
template <int D, bool UPDATE>
__global__ __launch_bounds__(256) void f32_attention_kernel(
    const char *__restrict__ blob, const float *__restrict__ qbuf, const float *kc,
    const float *vc, float *__restrict__ out, int heads, int slots, float scale, KvUpdateArgs up) {
  constexpr int U = 4;             // passes in flight
  constexpr int KV = D / 32;       // 16-byte pieces of a key per lane
  constexpr int KP = 256 / 8;      // keys of a score pass
  constexpr int VL = D / 4, G = 256 / VL;  // lanes of a value row, rows of a pass
  extern __shared__ __attribute__((aligned(16))) float sc[];  // scores [slots], then partial outputs [G][D]
  __shared__ float shf[4];
  __shared__ double shd[4];
  __shared__ __attribute__((aligned(16))) float own[UPDATE ? 3 : 1][UPDATE ? D : 1];  // q, k, v of the token
  const int t = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x;
  const BatchView bv = batch_view(blob);
  const ffmi_token_info tk = bv.tokens[t];
  const int Hl = heads * D;
  const int mine = UPDATE ? tk.store_slot : -1;  // the slot whose key and value are in LDS
  if constexpr (UPDATE) {
    if (tid < D / 2) {
      const KvUpdateF32 u = f32_kv_update(tk, t, hd, tid, up.qkv, up.rope, up.max_rope_pos, up.kc, up.vc, up.stage,
                                          heads, D, slots);
      own[0][tid] = u.q0, own[0][tid + D / 2] = u.q1;
      own[1][tid] = u.k0, own[1][tid + D / 2] = u.k1;
      own[2][tid] = u.va, own[2][tid + D / 2] = u.vb;
    }
    __syncthreads();
  }
  int kv_end = max(tk.prefix_len, tk.tree_len > 0 ? tk.tree_base + tk.tree_len : 0);
  kv_end = min(kv_end, slots);
  const float *K = kc + ((size_t)tk.req * heads + hd) * slots * D;
  const float *V = vc + ((size_t)tk.req * heads + hd) * slots * D;
  const float NEG = -3.402823466e38f;
  const int sub = tid & 7;
  f4 q[KV];
#pragma unroll
  for (int i = 0; i < KV; ++i)
    q[i] = UPDATE ? *reinterpret_cast<const f4 *>(&own[0][(i * 8 + sub) * 4])
                  : *reinterpret_cast<const f4 *>(qbuf + (size_t)t * Hl + hd * D + (i * 8 + sub) * 4);
  float mx = NEG;
  for (int j0 = 0; j0 < kv_end; j0 += U * KP) {
    f4 k[U][KV];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // (past the end: the last key again, dropped)
      const float *kr = K + (size_t)min(j0 + u * KP + (tid >> 3), kv_end - 1) * D + sub * 4;
#pragma unroll
      for (int i = 0; i < KV; ++i) k[u][i] = *reinterpret_cast<const f4 *>(kr + i * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * KP + (tid >> 3);
      float acc = 0.f;
      if (UPDATE && j == mine)
#pragma unroll
        for (int i = 0; i < KV; ++i) k[u][i] = *reinterpret_cast<const f4 *>(&own[1][(i * 8 + sub) * 4]);
#pragma unroll
      for (int i = 0; i < KV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __fadd_rn(acc, __fmul_rn(q[i][e], k[u][i][e]));
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) acc = __fadd_rn(acc, __shfl_xor(acc, off));
      const unsigned jj = (unsigned)(j - tk.tree_base);
      const bool vis = j < kv_end && (j < tk.prefix_len || (jj < (unsigned)tk.tree_len &&
                                                            ((tk.tree_vis >> (jj & 63)) & 1ull)));
      const float sv = __fmul_rn(scale, acc);
      if (vis) mx = fmaxf(mx, sv);
      if (sub == 0 && j < kv_end) sc[j] = vis ? sv : __builtin_nanf("");  // NaN: an invisible key
    }
  }
  mx = block_reduce256(mx, shf, [](float p, float r) { return fmaxf(p, r); });
  double sum = 0.0;
  for (int j = tid; j < kv_end; j += 256) {
    const float sv = sc[j];
    const float e = sv == sv ? expf(__fsub_rn(sv, mx)) : 0.f;
    sc[j] = e;
    sum += (double)e;
  }
  sum = block_reduce256(sum, shd, [](double p, double r) { return p + r; });
  const float inv = __fdiv_rn(1.0f, __fadd_rn((float)sum, 1e-6f));
  // P.V: group gi takes keys gi, gi + G, ...; its lane i elements 4 i .. 4 i + 3
  const int gi = tid / VL, i = tid % VL;
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  for (int j0 = gi; j0 < kv_end; j0 += U * G) {
    f4 v[U];
    float p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = min(j0 + u * G, kv_end - 1);
      v[u] = *reinterpret_cast<const f4 *>(V + (size_t)j * D + i * 4);
      if (UPDATE && j == mine) v[u] = *reinterpret_cast<const f4 *>(&own[2][i * 4]);
      p[u] = j0 + u * G < kv_end ? sc[j] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p[u] != 0.f)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = __fadd_rn(acc[e], __fmul_rn(__fmul_rn(p[u], inv), v[u][e]));
  }
  __syncthreads();  // the scores are read
  *reinterpret_cast<f4 *>(&sc[gi * D + i * 4]) = acc;
  __syncthreads();
  if (tid < D) {
    float o = sc[tid];
#pragma unroll
    for (int r = 1; r < G; ++r) o = __fadd_rn(o, sc[r * D + tid]);
    out[(size_t)t * Hl + hd * D + tid] = o;
  }
}

template <bool UPDATE>
static hipError_t run_attention_f32(const char *blob, int T, const float *qbuf, const float *kc, const float *vc,
                                    float *out, int heads, int d, int slots, float scale, const KvUpdateArgs &up,
                                    hipStream_t s) {
  const size_t lds = (size_t)std::max(slots, 1024) * sizeof(float);  // (partial outputs: 1024)
  if ((size_t)(d + 256 + slots) * sizeof(float) > 64 * 1024) return hipErrorInvalidValue;
  const dim3 grid(T, heads), block(256);
#define FFMI_ATTN_F32(DD)                                                                                             \
  hipLaunchKernelGGL((f32_attention_kernel<DD, UPDATE>), grid, block, lds, s, blob, qbuf, kc, vc, out, heads, slots, \
                     scale, up)
  if (d == 128) FFMI_ATTN_F32(128);
  else if (d == 64) FFMI_ATTN_F32(64);
  else if (d == 32) FFMI_ATTN_F32(32);
  else return hipErrorInvalidValue;
#undef FFMI_ATTN_F32
  return hipGetLastError();
}

hipError_t launch_attention_f32(const char *blob, int T, const float *qbuf, const float *kc,
                                const float *vc, float *out, int heads, int d, int slots,
                                float scale, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  return run_attention_f32<false>(blob, T, qbuf, kc, vc, out, heads, d, slots, scale, KvUpdateArgs(), s);
}

hipError_t launch_update_attention_f32(const char *blob, int T, int C, const float *qkv, const float *rope,
                                       int max_rope_pos, float *qbuf, float *kc, float *vc, float *stage, float *out,
                                       int heads, int d, int slots, float scale, bool distinct, hipStream_t s) {
  // (beside the scores: the token's rows and the reductions, 2 KiB)
  const bool one = distinct && (size_t)std::max(slots, 1024) * sizeof(float) + 2048 <= 64 * 1024;
  const hipError_t e = launch_kv_update_f32(blob, one ? 0 : T, C, qkv, rope, max_rope_pos, qbuf, kc, vc, stage, heads,
                                            d, slots, s);
  if (e != hipSuccess || T <= 0) return e;
  if (!one) return launch_attention_f32(blob, T, qbuf, kc, vc, out, heads, d, slots, scale, s);
  KvUpdateArgs up;
  up.qkv = qkv, up.rope = rope, up.max_rope_pos = max_rope_pos, up.kc = kc, up.vc = vc, up.stage = stage;
  return run_attention_f32<true>(blob, T, qbuf, kc, vc, out, heads, d, slots, scale, up, s);
}

// ---------------------------------------------------------------------------
// softmax + argmax / arg-top-k on fp32 probabilities: p_i = expf(z_i - max) /
// (float)sum (sum in fp64); k rounds of a block arg-max under the order
// (p desc, index asc), each round taking the first element after the
// previous pick in that order (arg_topk.cu:208-330 ties: lower index first).
// ---------------------------------------------------------------------------
// NV > 0: the row (V <= NV * 1024) is read once, all loads in flight together,
// and kept in registers; NV == 0: any V, read per pass.
template <int NV>
__global__ __launch_bounds__(1024) void f32_softmax_topk_kernel(const float *__restrict__ logits,
                                                               int V, int ld, int k,
                                                               int32_t *__restrict__ ids,
                                                               float *__restrict__ probs) {
  __shared__ float shf[16];
  __shared__ double shd[16];
  __shared__ float sp[16];
  __shared__ int si[16];
  const int t = blockIdx.x, tid = threadIdx.x, nw = blockDim.x >> 6;
  const float *z = logits + (size_t)t * ld;
  float zr[NV ? NV : 1];
#pragma unroll
  for (int j = 0; j < NV; ++j) zr[j] = z[min(tid + j * 1024, V - 1)];
  // f(i, z_i) for this thread's elements, ascending
  auto each = [&](auto f) {
    if constexpr (NV > 0) {
#pragma unroll
      for (int j = 0; j < NV; ++j)
        if (tid + j * 1024 < V) f(tid + j * 1024, zr[j]);
    } else {
      for (int i = tid; i < V; i += 1024) f(i, z[i]);
    }
  };
  float mx = -3.402823466e38f;
  each([&](int, float v) { mx = fmaxf(mx, v); });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  if ((tid & 63) == 0) shf[tid >> 6] = mx;
  __syncthreads();
  mx = shf[0];
  for (int w = 1; w < nw; ++w) mx = fmaxf(mx, shf[w]);
  double sum = 0.0;
  each([&](int, float v) { sum += (double)expf(__fsub_rn(v, mx)); });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if ((tid & 63) == 0) shd[tid >> 6] = sum;
  __syncthreads();
  sum = shd[0];
  for (int w = 1; w < nw; ++w) sum += shd[w];
  const float s = (float)sum;
  float pprev = 3.402823466e38f;
  int iprev = -1;
  for (int r = 0; r < k; ++r) {
    float bp = -1.f, bz = -3.402823466e38f;
    int bi = V;
    each([&](int i, float v) {
      // a logit this far below the row's best (first round) or the thread's has
      // a smaller probability (exp is monotone to a few ulps): not evaluated
      if (v < (r == 0 ? mx : bz) - 1e-3f) return;
      const float p = __fdiv_rn(expf(__fsub_rn(v, mx)), s);
      const bool after = p < pprev || (p == pprev && i > iprev);
      if (after && (p > bp || (p == bp && i < bi))) bp = p, bi = i, bz = v;
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float op = __shfl_xor(bp, off);
      const int oi = __shfl_xor(bi, off);
      if (op > bp || (op == bp && oi < bi)) bp = op, bi = oi;
    }
    __syncthreads();  // sp / si of the previous round are consumed
    if ((tid & 63) == 0) sp[tid >> 6] = bp, si[tid >> 6] = bi;
    __syncthreads();
    bp = sp[0], bi = si[0];
    for (int w = 1; w < nw; ++w)
      if (sp[w] > bp || (sp[w] == bp && si[w] < bi)) bp = sp[w], bi = si[w];
    if (tid == 0) {
      ids[(size_t)t * k + r] = bi;
      probs[(size_t)t * k + r] = bp;
    }
    pprev = bp, iprev = bi;
  }
}

hipError_t launch_softmax_topk_f32(const float *logits, int T, int V, int k, int32_t *ids,
                                   float *probs, hipStream_t s, int ld) {
  if (T <= 0) return hipSuccess;
  if (ld == 0) ld = V;
  if (k < 1 || k > V || ld < V) return hipErrorInvalidValue;
  if (V <= 32 * 1024)
    hipLaunchKernelGGL(f32_softmax_topk_kernel<32>, dim3(T), dim3(1024), 0, s, logits, V, ld, k,
                       ids, probs);
  else
    hipLaunchKernelGGL(f32_softmax_topk_kernel<0>, dim3(T), dim3(1024), 0, s, logits, V, ld, k, ids,
                       probs);
  return hipGetLastError();
}

// Rows of logits as fp32, into pinned host memory: bound by PCIe, so what matters is
// whole lines in flight (a wave writes 1 KiB at a time) and that the host does not wait
// for the last row before it copies the first.  So a row's workgroups write one row after
// the other, and one that has written its columns of a row says so in a word of its own,
// there[row][blockIdx.x] = mark (no counters to clear, no workgroup waits for another).
// Up to 32 workgroups a row; short rows side by side, 32 workgroups in all (200 rows of 1000
// one after the other: whole steps 393 us, so 173).  Rows of dst are whole pieces of four,
// whatever V is (200 rows of 33001 in single words: 3290 us, so 870).
// With rows shared out over 2, 4 and 16 groups of workgroups they end later than one after
// the other: 24 decode steps of 8 rows of 32000, whole steps, 22.15 ms in one group, 22.18 in
// two, 22.40 and 22.53 in four and 16 (all rows copied after the kernel: 23.0).
template <class IN>
__global__ __launch_bounds__(256) void logit_rows_kernel(const IN *__restrict__ logits, size_t ld, LogitRowIds ids,
                                                         int n, int V, float *__restrict__ dst, uint32_t *there,
                                                         uint32_t mark) {
  typedef IN in4 __attribute__((ext_vector_type(4)));
  const bool wide = V % 4 == 0 && ld % 4 == 0;
  for (int row = blockIdx.y; row < n; row += gridDim.y) {
    const IN *src = logits + (size_t)ids.row[row] * ld;
    float *to = dst + (size_t)row * LogitRowIds::pitch(V);
    for (int i = (blockIdx.x * 256 + threadIdx.x) * 4; i < V; i += gridDim.x * 1024) {
      in4 v;
      if (wide) v = *reinterpret_cast<const in4 *>(src + i);
      else
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = src[min(i + j, V - 1)];
      *reinterpret_cast<f4 *>(to + i) = f4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    }
    // every wave's writes are there, then the word (a release for the host)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(there + row * LogitRowIds::kParts + blockIdx.x, mark, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

hipError_t launch_logit_rows(const void *logits, bool half, size_t ld, const LogitRowIds &ids, int n, int V,
                             float *dst, uint32_t *there, uint32_t mark, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n > LogitRowIds::kMax) return hipErrorInvalidValue;
  const int parts = LogitRowIds::parts(V);
  const dim3 grid(parts, std::min(n, LogitRowIds::kParts / parts));
  if (half)
    hipLaunchKernelGGL(logit_rows_kernel<_Float16>, grid, dim3(256), 0, s, (const _Float16 *)logits, ld, ids, n, V,
                       dst, there, mark);
  else
    hipLaunchKernelGGL(logit_rows_kernel<float>, grid, dim3(256), 0, s, (const float *)logits, ld, ids, n, V, dst,
                       there, mark);
  return hipGetLastError();
}

}  // namespace ffmi

// public kernel-level entries (include/ffmi.h)
extern "C" ffmi_status ffmi_linear_f32(const float *X, const float *W, float *Y, int T,
                                       int out_dim, int in_dim, ffmi_stream stream) {
  FFMI_CHECK(T >= 0 && out_dim > 0 && in_dim > 0, FFMI_ERR_INVALID);
  FFMI_CHECK(in_dim % 32 == 0, FFMI_ERR_UNSUPPORTED);
  FFMI_CHECK(T == 0 || (X && W && Y), FFMI_ERR_INVALID);
  FFMI_HIP(ffmi::launch_gemm_f32(X, W, Y, T, out_dim, in_dim, (hipStream_t)stream));
  return FFMI_OK;
}

extern "C" ffmi_status ffmi_rmsnorm_f32(const float *x, const float *w, float *out, int T, int H,
                                        float eps, ffmi_stream stream) {
  FFMI_CHECK(x && w && out && T >= 0 && H > 0, FFMI_ERR_INVALID);
  FFMI_HIP(ffmi::launch_rmsnorm_f32(x, nullptr, w, nullptr, out, T, H, eps, (hipStream_t)stream));
  return FFMI_OK;
}

extern "C" ffmi_status ffmi_residual_rmsnorm_f32(const float *x1, const float *x2, const float *w,
                                                 float *residual_out, float *out, int T, int H,
                                                 float eps, ffmi_stream stream) {
  FFMI_CHECK(x1 && x2 && w && residual_out && out && T >= 0 && H > 0, FFMI_ERR_INVALID);
  FFMI_HIP(ffmi::launch_rmsnorm_f32(x1, x2, w, residual_out, out, T, H, eps, (hipStream_t)stream));
  return FFMI_OK;
}

extern "C" ffmi_status ffmi_silu_mul_f32(const float *a, const float *b, float *out, size_t n,
                                         ffmi_stream stream) {
  FFMI_CHECK(a && b && out && n <= (size_t)INT32_MAX, FFMI_ERR_INVALID);
  FFMI_HIP(ffmi::launch_silu_mul_f32(a, b, out, 1, (int)n, n, n, (hipStream_t)stream));
  return FFMI_OK;
}

extern "C" ffmi_status ffmi_arg_topk_f32(const float *logits, int T, int V, int k, int32_t *ids,
                                         float *probs, ffmi_stream stream) {
  FFMI_CHECK(logits && ids && probs && T >= 0 && V > 0 && k >= 1 && k <= 4 && k <= V,
             FFMI_ERR_INVALID);
  FFMI_HIP(ffmi::launch_softmax_topk_f32(logits, T, V, k, ids, probs, (hipStream_t)stream));
  return FFMI_OK;
}
