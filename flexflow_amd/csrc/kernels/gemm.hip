// gemm.hip -- the fp16 GEMM entry points (kernels: gemm_kernels.h).
#include "gemm_kernels.h"

namespace ffmi {

size_t gemm_workspace_bytes(int T, int N, int K, int epilogue, bool aligned) {
  return gemm_slab_bytes(T, N, K, epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM), false, aligned);
}

hipError_t launch_partials_reduce(const Partials &p, uint16_t *Y, int T, int N, hipStream_t s) {
  if (T <= 0 || p.S <= 0) return hipSuccess;
  // (> 8: the per-head o-projection slabs of a small model, OprojArgs)
  if (p.S > 16 || p.NP % 16 || N > p.NP) return hipErrorInvalidValue;
  const long total = (long)T * ((N + 3) / 4);
  const unsigned blocks = (unsigned)((total + 255) / 256);
#define FFMI_PRED(MS)                                                                          \
  hipLaunchKernelGGL((gemm_reduce_kernel<0, MS>), dim3(blocks), dim3(256), 0, s, p.p, Y, T, N, \
                     p.NP / 16, p.S, 0, 0.f)
  if (p.S <= 2) FFMI_PRED(2);
  else if (p.S <= 4) FFMI_PRED(4);
  else if (p.S <= 8) FFMI_PRED(8);
  else FFMI_PRED(16);
#undef FFMI_PRED
  return hipGetLastError();
}

hipError_t launch_gemm(const uint16_t *X, const uint16_t *Wp, uint16_t *Y, float *ws,
                       size_t ws_bytes, int T, int N, int K, int epilogue, hipStream_t s,
                       Partials *defer, int wpitch, const FuseArgs *fuse) {
  if ((epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM)) == FFMI_EPI_SILU_MUL)
    return launch_gemm_kind<1>(X, Wp, Y, ws, ws_bytes, T, N, K, epilogue, s, defer, wpitch, fuse);
  return launch_gemm_kind<0>(X, Wp, Y, ws, ws_bytes, T, N, K, epilogue, s, defer, wpitch, fuse);
}

// FFMI_SUM_NORM=0: the norm is a launch of its own (A/B, tests; read per call)
bool gemm_sum_norm_fits(int T, int N, int K, int epilogue, const Partials &sums) {
  const char *e = getenv("FFMI_SUM_NORM");
  const bool paired = (epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM)) == FFMI_EPI_SILU_MUL;
  if (norm_fault() || (e && !atoi(e)) || T < 1 || T > kSumNormRows || N < 1 || K > kSumNormWidth || K % 32) return false;
  if (sums.S < 1 || sums.S > (paired ? 16 : 8) || sums.NP < K || sums.NP % 4) return false;
  // (its slabs could lie where it would write its own)
  return paired || skinny_split(T, N, K, 0, true) == 1;
}

hipError_t launch_gemm_sum_norm(const SumNormArgs &a, const uint16_t *Wp, uint16_t *Y, int T, int N, int K,
                                int epilogue, hipStream_t s) {
  if (!gemm_sum_norm_fits(T, N, K, epilogue, Partials{a.sums, a.S, a.NP}) || a.res_in == a.res_out)
    return hipErrorInvalidValue;
  const bool paired = (epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM)) == FFMI_EPI_SILU_MUL;
  const bool nt = (epilogue & FFMI_W_STREAM) != 0;
  const int KT = K / 32, ntiles = (N + 15) / 16, yp = epilogue & FFMI_Y_PACKED ? N : 0;
  if (yp && N % 32) return hipErrorInvalidValue;
  const size_t wts = w_tile_stride(KT), wks = w_k_stride(paired ? 2 * ntiles : ntiles);
  float *none = nullptr;
  const uint16_t *x = nullptr;
#define FFMI_MADE(NT, E, NL, FZ)                                                                                  \
  hipLaunchKernelGGL((gemm_skinny_kernel<1, NT, 4, 8, E, false, NL, FZ>), dim3(ntiles), dim3(256),                \
                     3 * NT * 4 * 64 * sizeof(float), s, x, Wp, Y, none, T, N, K, KT, NT * ntiles, 1, yp, wts, wks, a)
#define FFMI_MADE_NL(NT, E, FZ)          \
  do {                                   \
    if (nt) FFMI_MADE(NT, E, true, FZ);  \
    else FFMI_MADE(NT, E, false, FZ);    \
  } while (0)
  if (paired) {
    if (a.S <= 8) FFMI_MADE_NL(2, 1, 5);
    else if (a.S <= 12) FFMI_MADE_NL(2, 1, 6);
    else FFMI_MADE_NL(2, 1, 7);
  } else if (ntiles >= 1024) {  // (the wave kernel's, as in dispatch_nt)
    const dim3 grid(((ntiles + 1) / 2 + 3) / 4);
    if (nt)
      hipLaunchKernelGGL((gemm_wave_kernel<1, 2, 4, true, 4, 0, true>), grid, dim3(256), 0, s, x, Wp, Y, none, T, N,
                         KT, ntiles, 1, yp, wts, wks, a);
    else
      hipLaunchKernelGGL((gemm_wave_kernel<1, 2, 4, false, 4, 0, true>), grid, dim3(256), 0, s, x, Wp, Y, none, T, N,
                         KT, ntiles, 1, yp, wts, wks, a);
  } else {
    FFMI_MADE_NL(1, 0, 5);
  }
#undef FFMI_MADE_NL
#undef FFMI_MADE
  return hipGetLastError();
}

int gemm_tile_form(int T, int N, int K, int epilogue, int *slices) {
  const bool paired = (epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM)) == FFMI_EPI_SILU_MUL;
  *slices = 1;
  const bool xp = (epilogue & FFMI_X_PACKED) != 0;
  if (T <= 64 || K % 32) return -1;
  if (!use_tiles(T, N, K, paired, xp, false, false)) {
    const MidPlan m = mid_plan(T, N, K, paired);
    return takes_six(T, K, m.NTW, m.S, xp) ? kNumTileForms : -1;
  }
  const TilePlan p = tile_plan(T, N, K, paired, false, false);
  *slices = p.S;
  return p.form;
}

int gemm_few_rows_slices(int T, int N, int K) { return skinny_split(T, N, K, 0, true); }

// A k-step of row-major operands takes the tile kernel about 0.12 us longer, all of a
// slice's one after another: long slices, and unsplit ones on few CUs.  T = 257, M-split
// kernel (which split them) / tiles / packed and tiles: 2048 x 2048 16.8 / 21.0 / 16.2 us,
// 4096 x 2048 21.2 / 21.6 / 16.2, 1024 x 1024 10.8 / 12.2 / 10.8, 768 x 768 10.1 / 10.2 / 9.8; but 512 x 4096
// in 8 slices 14.0 / 12.6 / 15.4 and 4096 x 1376 14.0 / 12.5 / 12.9.
bool gemm_pack_pays(int T, int N, int K, int epilogue) {
  const bool paired = (epilogue & ~(FFMI_X_PACKED | FFMI_Y_PACKED | FFMI_W_STREAM)) == FFMI_EPI_SILU_MUL;
  if (T <= 64 || K % 32 || !use_tiles(T, N, K, paired, false, false, false)) return false;
  const TilePlan p = tile_plan(T, N, K, paired, false, false);
  const int steps = (K / 32 + p.S - 1) / p.S;
  return steps > 48 || (p.S == 1 && steps >= 24 && p.nbm * p.nbn <= 64);
}

// Packed activation tiles: Xp[mt][kt][lane][8] = X[mt*16 + (lane&15)][kt*32 + 8(lane>>4) + e]
// (rows >= T zero) -- the MFMA operand fragment order of the weights (weights.hip),
// so a GEMM reads each activation fragment as one contiguous 1 KiB.
// Whole 256-byte row pieces in, whole fragments out, turned round in LDS.
__global__ __launch_bounds__(256) void pack_act_kernel(const uint16_t *__restrict__ X,
                                                      uint16_t *__restrict__ Xp, int T, int K, int KT) {
  __shared__ uint4 tile[4][64];
  const int mt = blockIdx.y, kt0 = blockIdx.x * 4, i = threadIdx.x;
  const int r = mt * 16 + (i >> 4), k = kt0 * 32 + (i & 15) * 8;
  uint4 v = make_uint4(0, 0, 0, 0);
  if (r < T && k < K) v = *reinterpret_cast<const uint4 *>(X + (size_t)r * K + k);
  tile[(i >> 2) & 3][(i & 3) * 16 + (i >> 4)] = v;
  __syncthreads();
  const int kt = kt0 + (i >> 6);
  if (kt < KT)
    *reinterpret_cast<uint4 *>(Xp + (((size_t)mt * KT + kt) * 64 + (i & 63)) * 8) = tile[i >> 6][i & 63];
}

size_t packed_act_bytes(int T, int K) { return (size_t)((T + 15) / 16) * 16 * K * 2; }

hipError_t launch_pack_act(const uint16_t *X, uint16_t *Xp, int T, int K, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(pack_act_kernel, dim3((K / 32 + 3) / 4, (T + 15) / 16), dim3(256), 0, s, X, Xp, T, K,
                     K / 32);
  return hipGetLastError();
}

// diagnostics: stamps of the last FFMI_GEMM_STAMP launch (8 int64 per wave)
long gemm_debug_stamps(long long *dst, long max_waves) {
  long long *buf = stamp_buf();
  const long n = g_stamp_entries < max_waves ? g_stamp_entries : max_waves;
  if (!buf || n <= 0) return 0;
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (hipMemcpy(dst, buf, (size_t)n * 8 * sizeof(long long), hipMemcpyDeviceToHost) != hipSuccess)
    return -1;
  return n;
}

}  // namespace ffmi
