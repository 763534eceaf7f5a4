// attention.hip -- incremental / speculative / tree-verify attention on MFMA.
//
// One kernel family serves the reference's three attention ops, because on
// the device they differ only in WHICH cache slots a query may see:
//  * IncMultiHeadSelfAttention    (inc_multihead_self_attention.cu:372-623,
//    prompt path :98-366): keys [0, pos] (causal);
//  * TreeIncMultiHeadSelfAttention (tree_inc_multihead_self_attention.cu:
//    35-333): keys [0, non_tree_cache_size) plus tree slot j iff
//    causalMask.mask[j] has the query's bit (layer-order token tree);
//  * SpecIncMultiHeadSelfAttention (spec_inc_multihead_self_attention.cu:
//    36-309): same bitmask rule with the query's tree index as its bit.
// The host packs that rule per token (ffmi_token_info: prefix_len,
// tree_base/len/bit), so the kernel is mode-agnostic.  (The reference's
// `1 << qi` on a 32-bit int, tree_inc...cu:168-169, is done in 64 bits here.)
//
// KV-cache layout (handle-owned, MI355X-first): K[req][head][slot][d] and
// V^T[req][head][d][slot], slots = S + tree rounded up to 32.  With these two
// orientations both attention GEMMs read their MFMA operands straight from
// HBM as 16-B / 8-B vectors:
//   S^T[key][q] = K . Q^T        (A = K rows, B = Q rows)   16x16x32 f16
//   O^T[d][q]  += V^T . P^T      (A = V^T rows, B = P^T)    16x16x32 f16
// and the S^T accumulator of a lane (query q = lane&15, keys 4g..4g+3 of
// each 16-key half, g = lane>>4) IS the lane's P^T B-fragment under the key
// permutation k(g,j) = (j<4 ? 4g+j : 16+4g+j-4) -- no LDS transpose.  P is
// fed as an fp16 hi/lo pair (two MFMAs), which keeps ~22 bits of P, matching
// the reference's fp32 P.V accumulation (inc...cu:575-581) instead of
// rounding P to fp16.  Softmax follows the reference: __expf, running max,
// out = sum(e_j v_j) / (sum_j e_j + 1e-6)   (inc...cu:532-547).
//
// Work decomposition: one workgroup per (work item = <=16 queries of one
// request, head); its 8 waves stride over 32-key chunks with private online
// softmax state and merge through LDS.  Every key/value byte of a request is
// read once per 16-query tile (the reference's tree kernel re-reads the
// whole K/V once per query, tree_inc...cu:135).
#include <stdlib.h>

#include <algorithm>

#include "../ffmi_internal.h"

namespace ffmi {

__device__ __forceinline__ float h2f(uint16_t v) { return __half2float(__ushort_as_half(v)); }
__device__ __forceinline__ uint16_t f2h(float v) { return __half_as_ushort(__float2half_rn(v)); }

// commit_tokens_kernel (tree_inc...cu:335-396): accepted tokens of the
// previous verify batch move from the staging rows to their depth slot.
__global__ void commit_kernel(const char *__restrict__ blob, int C,
                              const uint16_t *__restrict__ stage, uint16_t *__restrict__ kc,
                              uint16_t *__restrict__ vc, int heads, int d, int slots) {
  const int item = blockIdx.x;  // commit * heads + head
  const int ci = item / heads, h = item % heads;
  if (ci >= C) return;
  BatchView bv = batch_view(blob);
  const ffmi_commit_info cm = bv.commits[ci];
  if (cm.depth < 0 || cm.depth >= slots) return;
  const int Hl = heads * d;
  const uint16_t *st = stage + (size_t)cm.src_token * 2 * Hl + h * d;
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    kc[(((size_t)cm.req * heads + h) * slots + cm.depth) * d + i] = st[i];
    vc[(((size_t)cm.req * heads + h) * d + i) * slots + cm.depth] = st[Hl + i];
  }
}

hipError_t launch_commit(const char *blob, int C, const uint16_t *stage, uint16_t *kc,
                         uint16_t *vc, int heads, int d, int slots, hipStream_t s) {
  if (C <= 0) return hipSuccess;
  hipLaunchKernelGGL(commit_kernel, dim3(C * heads), dim3(64), 0, s, blob, C, stage, kc, vc,
                     heads, d, slots);
  return hipGetLastError();
}

// Fused KV update of one step: RoPE (HF rotate-half, inc...cu:664-738) + KV
// store (store_kv_cache inc...cu:35-61 / update_tree_branch_kv_cache_fused
// tree_inc...cu:433-478 / spec_inc_store_kv_cache spec_inc...cu:311-358) +
// staging copy for the next step's commits, for one (attention work item =
// <= NQ consecutive tokens of a request, head).  Shared by kv_update_kernel
// and the FUSED attention prologue.
//  * a thread unit is 4 consecutive rotation pairs (d = i0..i0+3 and
//    i0+D/2..) of one token: 8-B fp16 or 16-B fp32-slab loads, 8-B stores;
//  * every load of a thread (all its units, all slabs) is issued before its
//    first store -- the update is a chain of dependent HBM round trips
//    otherwise (units past q_count load token 0 and store nothing);
//  * V goes through LDS so that V^T rows are written as runs of consecutive
//    slots instead of one 2-byte store per (token, d).
__device__ __forceinline__ f4 round_h4(f4 a) {  // fp16 value of the combined sum
  return f4{h2f(f2h(a[0])), h2f(f2h(a[1])), h2f(f2h(a[2])), h2f(f2h(a[3]))};
}
__device__ __forceinline__ void st_h4(uint16_t *p, uint16_t a, uint16_t b, uint16_t c,
                                      uint16_t d) {
  *reinterpret_cast<uint2 *>(p) = make_uint2(a | ((uint32_t)b << 16), c | ((uint32_t)d << 16));
}

// after_loads() runs once this thread's update loads are in flight (the
// fused attention issues its first K/V chunk there: loads complete in issue
// order, so anything issued BEFORE these would delay them).
// Tail mode (sKt != nullptr, the fused attention): K rows and V^T columns of
// the stored tokens also go to the workgroup's LDS tail tile (slot - tail0),
// where its attention reads them -- no wait for the global stores; V^T then
// goes to HBM from sVt.  before_stores() runs (in every thread) once the
// loads are back, before the first store.
// PSRC: 1 = qkv from split-K slabs, 0 = fp16 qkv, -1 = decided at run time
// by `part` (a compile-time source keeps the two load paths from joining:
// the join's register copies waited for half of the slab loads).
template <int D, int NQ, int NT, int PSRC = -1, class AfterLoads, class BeforeStores>
__device__ __forceinline__ void kv_update_item(
    const BatchView &bv, const WorkDev *__restrict__ wdp, int h, int heads, int slots, int T,
    const uint16_t *__restrict__ qkv, const float *__restrict__ part, int pS, int pNP,
    const float *__restrict__ rope, int max_rope_pos, uint16_t *__restrict__ qbuf,
    uint16_t *__restrict__ kc, uint16_t *__restrict__ stage_wr, uint16_t (*sV)[NQ + 1],
    int *sSlot, uint16_t (*sQ)[D + 8], uint16_t (*sKt)[D + 8],
    uint16_t (*sVt)[kTailSlots + 8], int tail0, AfterLoads &&after_loads,
    BeforeStores &&before_stores) {
  constexpr int HD = D / 2, G = HD / 4, UNITS = NQ * G, U = (UNITS + NT - 1) / NT;
  const int Hl = heads * D;
  const ffmi_attn_work w = wdp->w;
  // channels: 0 q lo, 1 q hi, 2 k lo, 3 k hi, 4 v lo, 5 v hi
  f4 x[U][6], y[U][6], cs[U][2];  // y: second fp32 slab
  int tslot[U], treq[U];  // (scalar fields: a struct copy would go to scratch)
  int tl[U], i0[U];
  // One round trip for every prologue load.  The RoPE positions of the
  // item's tokens come through the scalar cache (16 dwords of the work item,
  // lgkmcnt; readfirstlane keeps them there -- the per-lane select over them
  // was folded into a vector load), so the RoPE-row loads do not wait on any
  // vector load; the qkv
  // slabs (addresses known up front), the RoPE rows and the token records
  // then go out back to back.  (Vector loads complete in issue order: with
  // the positions loaded per lane, the RoPE rows waited for that load and
  // for everything issued before it.)
  const uint32_t *rp32 = reinterpret_cast<const uint32_t *>(wdp->rope_pos);
  uint32_t rpw[FFMI_ATTN_QTILE / 2];
#pragma unroll
  for (int j = 0; j < FFMI_ATTN_QTILE / 2; ++j) rpw[j] = __builtin_amdgcn_readfirstlane(rp32[j]);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = min((int)threadIdx.x + u * NT, UNITS - 1);
    tl[u] = e / G, i0[u] = (e % G) * 4;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int t = w.q_start + (tl[u] < w.q_count ? tl[u] : 0);
    const int col[6] = {h * D + i0[u], h * D + i0[u] + HD, Hl + h * D + i0[u],
                        Hl + h * D + i0[u] + HD, 2 * Hl + h * D + i0[u],
                        2 * Hl + h * D + i0[u] + HD};
    if (PSRC == 1 || (PSRC < 0 && part)) {  // slabs 0 and 1 (slab 0 again when pS == 1: no branch)
      const float *p1 = part + (pS > 1 ? (size_t)T * pNP : 0);
#pragma unroll
      for (int c = 0; c < 6; ++c)
        x[u][c] = *reinterpret_cast<const f4 *>(part + (size_t)t * pNP + col[c]);
#pragma unroll
      for (int c = 0; c < 6; ++c)
        y[u][c] = *reinterpret_cast<const f4 *>(p1 + (size_t)t * pNP + col[c]);
    } else {  // raw fp16 bits now, converted after every load is out
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const uint2 r = *reinterpret_cast<const uint2 *>(qkv + (size_t)t * 3 * Hl + col[c]);
        y[u][c] = f4{__uint_as_float(r.x), __uint_as_float(r.y), 0.f, 0.f};
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int q = tl[u] < w.q_count ? tl[u] : 0;
    uint32_t wd = rpw[0];
#pragma unroll
    for (int j = 1; j < FFMI_ATTN_QTILE / 2; ++j) wd = (q >> 1) == j ? rpw[j] : wd;
    const int p = min((int)((q & 1) ? (wd >> 16) : (wd & 0xffffu)), max_rope_pos - 1);
    const f4 *r = reinterpret_cast<const f4 *>(rope + ((size_t)p * HD + i0[u]) * 2);
    cs[u][0] = r[0];  // c0 s0 c1 s1
    cs[u][1] = r[1];  // c2 s2 c3 s3
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int t = w.q_start + (tl[u] < w.q_count ? tl[u] : 0);
    tslot[u] = bv.tokens[t].store_slot;
    treq[u] = bv.tokens[t].req;
  }
  after_loads();
  // every prologue load is in flight before any of them is consumed: left
  // alone the scheduler summed the slabs right after they were issued and
  // gave their registers to the RoPE rows, so each group of loads waited for
  // the one before it (four round trips instead of one)
  __builtin_amdgcn_sched_barrier(0);
  if (PSRC == 0 || (PSRC < 0 && !part))
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const uint32_t a = __float_as_uint(y[u][c][0]), b = __float_as_uint(y[u][c][1]);
        x[u][c] = f4{h2f(a & 0xffff), h2f(a >> 16), h2f(b & 0xffff), h2f(b >> 16)};
      }
  if (PSRC == 1 || (PSRC < 0 && part)) {  // slabs in slice order, then fp16 (partials_value)
    if (pS > 1)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < 6; ++c) x[u][c] += y[u][c];
    const size_t slab = (size_t)T * pNP;
    for (int sl = 2; sl < pS; ++sl)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = w.q_start + (tl[u] < w.q_count ? tl[u] : 0);
        const int col[6] = {h * D + i0[u], h * D + i0[u] + HD, Hl + h * D + i0[u],
                            Hl + h * D + i0[u] + HD, 2 * Hl + h * D + i0[u],
                            2 * Hl + h * D + i0[u] + HD};
#pragma unroll
        for (int c = 0; c < 6; ++c)
          x[u][c] += *reinterpret_cast<const f4 *>(part + sl * slab + (size_t)t * pNP + col[c]);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 6; ++c) x[u][c] = round_h4(x[u][c]);
  }

  before_stores();
  // ---- stores
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (tl[u] >= w.q_count || (int)threadIdx.x + u * NT >= UNITS) continue;
    const int t = w.q_start + tl[u];
    uint16_t qlo[4], qhi[4], klo[4], khi[4], vlo[4], vhi[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float c = cs[u][j >> 1][(j & 1) * 2], sn = cs[u][j >> 1][(j & 1) * 2 + 1];
      const float qa = x[u][0][j], qb = x[u][1][j], ka = x[u][2][j], kb = x[u][3][j];
      qlo[j] = f2h(__fsub_rn(__fmul_rn(qa, c), __fmul_rn(qb, sn)));
      qhi[j] = f2h(__fadd_rn(__fmul_rn(qa, sn), __fmul_rn(qb, c)));
      klo[j] = f2h(__fsub_rn(__fmul_rn(ka, c), __fmul_rn(kb, sn)));
      khi[j] = f2h(__fadd_rn(__fmul_rn(ka, sn), __fmul_rn(kb, c)));
      vlo[j] = f2h(x[u][4][j]);
      vhi[j] = f2h(x[u][5][j]);
    }
    // rotated q: to LDS for the same workgroup's attention (fused), else HBM
    uint16_t *qo = sQ ? &sQ[tl[u]][i0[u]] : qbuf + (size_t)t * Hl + h * D + i0[u];
    st_h4(qo, qlo[0], qlo[1], qlo[2], qlo[3]);
    st_h4(qo + HD, qhi[0], qhi[1], qhi[2], qhi[3]);
    const bool store = tslot[u] >= 0 && tslot[u] < slots;
    if (store) {
      uint16_t *kr = kc + (((size_t)treq[u] * heads + h) * slots + tslot[u]) * D + i0[u];
      st_h4(kr, klo[0], klo[1], klo[2], klo[3]);
      st_h4(kr + HD, khi[0], khi[1], khi[2], khi[3]);
    }
    if (i0[u] == 0) sSlot[tl[u]] = store ? tslot[u] : -1;
    if (sKt) {  // (host-checked: every stored slot lies in the tail)
      if (store) {
        const int ts = tslot[u] - tail0;
        st_h4(&sKt[ts][i0[u]], klo[0], klo[1], klo[2], klo[3]);
        st_h4(&sKt[ts][i0[u] + HD], khi[0], khi[1], khi[2], khi[3]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sVt[i0[u] + j][ts] = vlo[j];
          sVt[i0[u] + HD + j][ts] = vhi[j];
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sV[i0[u] + j][tl[u]] = vlo[j];
        sV[i0[u] + HD + j][tl[u]] = vhi[j];
      }
    }
    if (stage_wr) {
      uint16_t *st = stage_wr + (size_t)t * 2 * Hl + h * D + i0[u];
      st_h4(st, klo[0], klo[1], klo[2], klo[3]);
      st_h4(st + HD, khi[0], khi[1], khi[2], khi[3]);
      st_h4(st + Hl, vlo[0], vlo[1], vlo[2], vlo[3]);
      st_h4(st + Hl + HD, vhi[0], vhi[1], vhi[2], vhi[3]);
    }
  }
}

// V^T[req][h][d][slot] rows from the LDS tile: lanes run over consecutive
// tokens of a d-row (call after a barrier that follows kv_update_item)
template <int D, int NQ>
__device__ __forceinline__ void kv_store_vt(const ffmi_attn_work &w, int h, int heads, int slots,
                                            uint16_t *__restrict__ vc,
                                            const uint16_t (*sV)[NQ + 1], const int *sSlot) {
  uint16_t *vt = vc + ((size_t)w.req * heads + h) * D * slots;
  for (int e = threadIdx.x; e < D * NQ; e += blockDim.x) {
    const int dd = e / NQ, tt = e % NQ;
    if (tt >= w.q_count) continue;
    const int sl = sSlot[tt];
    if (sl >= 0) vt[(size_t)dd * slots + sl] = sV[dd][tt];
  }
}

// Standalone KV update (items with more tokens than one attention launch
// should carry in its prologue): one workgroup per (item, head), one thread
// per unit, plus the TREE commits of the previous verify batch in extra
// blocks.  Commits read the OTHER half of the ping-pong staging (stage_rd)
// than the one this step writes (stage_wr), so both run in one launch; the
// host launches commits separately first when a commit depth coincides with
// a slot this step stores (the reference's commit-then-store order).
template <int D>
__global__ __launch_bounds__(FFMI_ATTN_QTILE * D / 8) void kv_update_kernel(
    const char *__restrict__ blob, int T, int W, int C, const uint16_t *__restrict__ qkv,
    const float *__restrict__ part, int pS, int pNP, uint16_t *__restrict__ qbuf,
    uint16_t *__restrict__ kc, uint16_t *__restrict__ vc, uint16_t *__restrict__ stage_wr,
    const uint16_t *__restrict__ stage_rd, const float *__restrict__ rope, int heads, int slots,
    int max_rope_pos) {
  constexpr int NQ = FFMI_ATTN_QTILE;
  constexpr int NT = NQ * D / 8;
  __shared__ uint16_t sV[D][NQ + 1];
  __shared__ int sSlot[NQ];
  const int Hl = heads * D;
  const BatchView bv = batch_view(blob);
  const int item = blockIdx.x / heads, h = blockIdx.x % heads;
  if (item >= W) {  // ---- commit block (tree_inc...cu:335-396)
    const int ci = item - W;
    if (ci >= C) return;
    const ffmi_commit_info cm = bv.commits[ci];
    if (cm.depth < 0 || cm.depth >= slots) return;
    const uint16_t *st = stage_rd + (size_t)cm.src_token * 2 * Hl + h * D;
    const int i = threadIdx.x;
    if (i < D) {
      kc[(((size_t)cm.req * heads + h) * slots + cm.depth) * D + i] = st[i];
      vc[(((size_t)cm.req * heads + h) * D + i) * slots + cm.depth] = st[Hl + i];
    }
    return;
  }
  const ffmi_attn_work w = bv.work[item].w;
  kv_update_item<D, NQ, NT>(bv, &bv.work[item], h, heads, slots, T, qkv, part, pS, pNP, rope,
                            max_rope_pos, qbuf, kc, stage_wr, sV, sSlot, nullptr, nullptr, nullptr,
                            0, [] {}, [] {});
  __syncthreads();
  kv_store_vt<D, NQ>(w, h, heads, slots, vc, sV, sSlot);
}

hipError_t launch_kv_update(const char *blob, int T, int W, int C, const uint16_t *qkv,
                            Partials qkvp, uint16_t *qbuf, uint16_t *kc, uint16_t *vc,
                            uint16_t *stage_wr, const uint16_t *stage_rd, const float *rope,
                            int heads, int d, int slots, int max_rope_pos, hipStream_t s) {
  if (W <= 0 && C <= 0) return hipSuccess;
  const dim3 grid((W + C) * heads);
  const float *pp = qkvp.S > 0 ? qkvp.p : nullptr;
  if (d == 128)
    hipLaunchKernelGGL(kv_update_kernel<128>, grid, dim3(FFMI_ATTN_QTILE * 16), 0, s, blob, T, W, C, qkv, pp,
                       qkvp.S, qkvp.NP, qbuf, kc, vc, stage_wr, stage_rd, rope, heads, slots,
                       max_rope_pos);
  else if (d == 64)
    hipLaunchKernelGGL(kv_update_kernel<64>, grid, dim3(FFMI_ATTN_QTILE * 8), 0, s, blob, T, W, C, qkv, pp,
                       qkvp.S, qkvp.NP, qbuf, kc, vc, stage_wr, stage_rd, rope, heads, slots,
                       max_rope_pos);
  else if (d == 32)  // (incremental decoding only: ffmi_attn_create)
    hipLaunchKernelGGL(kv_update_kernel<32>, grid, dim3(FFMI_ATTN_QTILE * 4), 0, s, blob, T, W, C, qkv, pp,
                       qkvp.S, qkvp.NP, qbuf, kc, vc, stage_wr, stage_rd, rope, heads, slots,
                       max_rope_pos);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// visibility from registers only: prefix range + the query's 64-bit tree word
__device__ __forceinline__ bool key_visible(int slot, int prefix_len, int tree_base,
                                            int tree_len, uint64_t tree_vis) {
  const unsigned j = (unsigned)(slot - tree_base);
  const bool in_tree = j < (unsigned)tree_len && ((tree_vis >> (j & 63)) & 1ull);
  return (slot < prefix_len) | in_tree;  // no branches: one select per key
}

// the larger of a lane's x and lane ^ 16's (32's): a row exchange in the register
// file; __shfl_xor goes through LDS
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// One 32-key chunk [base, base + 32) of a wave's query tiles: scores, running max
// and sum, weighted values.  Lane (qi, g) holds query 16 qt + qi and keys
// base + 8 g .. + 7; seen: slots below it are visible to the lane's query.
template <int D, int QT>
__device__ __forceinline__ void attn_chunk(int base, int g, const h8 (&kf)[2][D / 32],
                                           const h8 (&va)[D / 16], const h8 (&qf)[QT][D / 32],
                                           const bool (&qvalid)[QT], const int (&seen)[QT],
                                           const int (&pre)[QT], const int (&tb)[QT],
                                           const int (&tlen)[QT], const uint64_t (&tv)[QT],
                                           int kv_len, float scale, float (&m_run)[QT],
                                           float (&l_run)[QT], f4 (&o)[QT][D / 16]) {
  constexpr int KS = D / 32, DT = D / 16;
  const float NEG = -INFINITY;
  // S^T = K . Q^T: this lane holds query qt*16+qi, keys base + 8 g + 4 sub + r
  float sc[QT][8];
  bool hidden = false;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      f4 s = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[sub][ks], qf[qt][ks], s, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[qt][4 * sub + r] = __fmul_rn(scale, s[r]);
    }
    hidden |= base + 32 > seen[qt];
  }
  // a chunk that every query sees needs no masks (all but a prompt item's last
  // two): with them this was most of the instructions of a chunk.  A hidden
  // key's score becomes -inf, whose weight is 0.
  if (__any(hidden)) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int slot = base + 8 * g + j;
        const bool vis = qvalid[qt] && slot < kv_len && key_visible(slot, pre[qt], tb[qt], tlen[qt], tv[qt]);
        sc[qt][j] = vis ? sc[qt][j] : NEG;
      }
  }
  float m_new[QT], m_use[QT];
  bool moved = false;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float cmax = NEG;
#pragma unroll
    for (int j = 0; j < 8; ++j) cmax = fmaxf(cmax, sc[qt][j]);
    cmax = max_xor32(max_xor16(cmax));
    m_new[qt] = fmaxf(m_run[qt], cmax);
    m_use[qt] = (m_new[qt] == NEG) ? 0.f : m_new[qt];
    moved |= m_new[qt] != m_run[qt];
  }
  if (__any(moved)) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const float alpha = (m_run[qt] == NEG) ? 0.f : __expf(m_run[qt] - m_use[qt]);
      l_run[qt] *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[qt][t] *= alpha;
      m_run[qt] = m_new[qt];
    }
  }
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    h8 phi, plo;
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = __expf(sc[qt][j] - m_use[qt]);
      psum += e;
      const _Float16 hi = (_Float16)e;
      phi[j] = hi;
      plo[j] = (_Float16)(e - (float)hi);
    }
    l_run[qt] += psum;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      o[qt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[t], phi, o[qt][t], 0, 0, 0);
      o[qt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[t], plo, o[qt][t], 0, 0, 0);
    }
  }
}

// Item and head of a workgroup of a W x heads grid: those of one head, and in it
// of one request, lie on one XCD (workgroup ids go round the 8 XCDs), whose L2
// then holds the K/V that they share.  Ids in grid order, every XCD read all K/V:
// 33
// prompt items x 16 heads at about 1500 keys 60 us, 49 so.
__device__ __forceinline__ void attn_place(int &item, int &head, int W, int heads) {
  const int lin = (int)(blockIdx.y * gridDim.x + blockIdx.x), total = W * heads;
  const int xcd = lin & 7, per = total >> 3, rem = total & 7;
  const int at = xcd * per + min(xcd, rem) + (lin >> 3);
  item = at % W, head = at / W;
}

// Arguments of the fused prologue (FUSED kernels only; see attention_kernel).
struct KvUpdateArgs {
  int T, C;
  const uint16_t *qkv;
  const float *part;
  int pS, pNP;
  uint16_t *stage_wr;
  const uint16_t *stage_rd;
  const float *rope;
  int max_rope_pos;
  long long *stamps;  // ST kernels: per-wave timeline (diagnostics)
  // ZS kernels: per (request, head) and sharing workgroup (at most zmax) the partial
  // output [D] and its max and sum, and per (request, head) the count of partials
  // that are there (zero between launches).  (By request, not by item: steps of
  // different requests may run side by side.)
  float *zpart;
  unsigned *zcount;
  int zmax;
};

// One workgroup per (work item = <= 16*QT consecutive queries of a request,
// head); NW = 8 waves (two per SIMD: each hides the other's load latency)
// stride over 32-key chunks with private online-softmax state
// and merge through LDS.  QT query tiles share every K / V^T fragment load.
//
// FUSED (host-checked: each request has exactly one work item this step, as
// in decode, SSM beam steps and tree verify): the workgroup first applies its
// own request's TREE commits and the KV update of its own tokens for its
// head (kv_update_kernel's work), makes them visible to the workgroup, then
// attends -- one launch per step instead of two.
//
// OP (FUSED, QT == 1; OprojArgs in ffmi_internal.h): the workgroup also
// multiplies its rounded output rows by its head's K-slice of Wo (MFMA with
// the packed weight block as the A operand and the output rows, from LDS, as
// B -- the S^T = K.Q^T arrangement) and stores the fp32 product as slab
// `head`.  The slice is loaded after the key loop, so the merge hides its
// latency; wave w owns column tiles w, w + NW, ... (N <= 16 * 8 * NW).
//
// QS == 2 (FUSED, QT == 1; grids with CUs to spare: TP >= 2 verify steps,
// <= 128 (request, head) pairs): the item's queries are split over two
// workgroups (blockIdx.z = which 16), each running the whole item's commits
// and KV update -- the same values to the same addresses, and every K/V it
// reads from memory is below the tail, which neither writes -- and attending
// its own 16: the key loop and merge work per workgroup halve.  Per query the
// arithmetic is the QT == 2 kernel's (MFMA columns are independent), so the
// output is bit-identical.
// ZS (steps of one query per request, long contexts, few workgroups; attn_kv_split):
// gridDim.z workgroups share an item's chunks, each leaves its partial output, and the
// last one to arrive merges them -- no workgroup waits for another.  All of them run
// the item's KV update, the same values to the same addresses.
template <int D, int QT, int NW, bool FUSED, bool ST = false, int PSRC = -1, bool OP = false,
          int QS = 1, bool ZS = false>
__global__ __launch_bounds__(64 * NW, 1) void attention_kernel(
    const char *__restrict__ blob, uint16_t *__restrict__ qbuf, uint16_t *__restrict__ kc,
    uint16_t *__restrict__ vc, uint16_t *__restrict__ out, int heads, int slots, float scale,
    int out_packed, KvUpdateArgs kv, OprojArgs opa) {
  static_assert(!OP || (FUSED && QT == 1 && QS == 1), "output projection: fused, one query tile");
  static_assert(QS == 1 || (FUSED && QT == 1 && QS == 2), "query split: fused, 2 x 16 queries");
  static_assert(!ZS || (FUSED && QT == 1 && QS == 1 && !OP && D / 16 <= NW), "key split: fused, one query");
  constexpr int KS = D / 32;  // k-steps of the QK^T product
  constexpr int DT = D / 16;  // d-tiles of the PV product
  constexpr int NQ = 16 * QT;   // queries this workgroup attends
  constexpr int NQK = NQ * QS;  // tokens of the item (commits, KV update)
  int item = blockIdx.x, h = blockIdx.y;
  if (!FUSED) attn_place(item, h, (int)gridDim.x, (int)gridDim.y);
  const int qbase = QS > 1 ? (int)blockIdx.z * NQ : 0;
  constexpr int TS = kTailSlots;
  __shared__ float sm_m[NW][NQ];
  __shared__ float sm_l[NW][NQ];
  // the merge buffer shares its LDS with the FUSED tail tile (K rows and V^T
  // columns of slots [tail0, tail0 + TS)); a barrier separates their uses
  constexpr int SMO_BYTES = NW * QT * DT * 4 * 64 * 4;
  constexpr int TAIL_BYTES = FUSED ? (TS * (D + 8) + D * (TS + 8)) * 2 : 0;
  __shared__ __attribute__((aligned(16)))
  char smem[SMO_BYTES > TAIL_BYTES ? SMO_BYTES : TAIL_BYTES];
  auto sm_o = reinterpret_cast<float(*)[QT][DT][4][64]>(smem);
  auto sKt = reinterpret_cast<uint16_t(*)[D + 8]>(smem);
  auto sVt = reinterpret_cast<uint16_t(*)[TS + 8]>(smem + TS * (D + 8) * 2);

  // ST: lane 0 of each wave stores its timeline straight to kv.stamps
  long long *stp = nullptr;
  if (ST && kv.stamps && (threadIdx.x & 63) == 0)
    stp = kv.stamps + ((size_t)(blockIdx.y * gridDim.x + blockIdx.x) * NW + (threadIdx.x >> 6)) * 12;
  auto stamp = [&](int i) {
    if (ST && stp) stp[i] = __builtin_amdgcn_s_memrealtime();
  };
  stamp(0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qi = lane & 15;
  const int g = lane >> 4;
  const BatchView bv = batch_view(blob);
  // (fields, not a copy of the WorkDev: a private copy of its rope_pos array
  // would be indexed per lane and live in scratch)
  const ffmi_attn_work w = bv.work[item].w;
  const int Hl = heads * D;
  const uint16_t *kbase = kc + ((size_t)w.req * heads + h) * slots * D;
  const uint16_t *vbase = vc + ((size_t)w.req * heads + h) * D * slots;
  // K rows and V^T columns of one 32-key chunk: row m of score tile sub is key
  // 8 (m / 4) + 4 sub + m % 4, so the lane that gets scores 4 g + r of both
  // tiles holds keys 8 g .. 8 g + 7 and its V^T operand is 16 bytes of each row
  // (keys in row order: two 8-byte loads, half the bytes of each line used at a
  // time) (chunk indices are clamped by
  // the caller: the cache is allocated to a multiple of 32 slots)
  const int krow0 = 8 * (qi >> 2) + (qi & 3);
  auto load_keys = [&](int c, h8 (&kf)[2][KS]) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const uint16_t *krow = kbase + (size_t)(c * 32) * D + (krow0 + 4 * sub) * D + 8 * g;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[sub][ks] = *reinterpret_cast<const h8 *>(krow + 32 * ks);
    }
  };
  auto load_values = [&](int c, h8 (&va)[DT]) {
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const uint16_t *vt = vbase + (size_t)t * 16 * slots + c * 32;
      va[t] = *reinterpret_cast<const h8 *>(vt + (lane & 15) * slots + 8 * g);
    }
  };
  auto load_chunk = [&](int c, h8 (&kf)[2][KS], h8 (&va)[DT]) {
    load_keys(c, kf);
    load_values(c, va);
  };
  // FUSED: every slot this step writes for the request (its stores and TREE
  // commits) lies in the LDS tail [tail0, kv_len) (host-checked, lds_tail);
  // the keys below tail0 are untouched this step, so their chunks load from
  // HBM at any time and a wave's first one goes out with the prologue's
  // loads.  The tail's chunks are read from LDS: the prologue writes the new
  // K/V there as well as to HBM, and the attention never waits for its own
  // global stores.
  const int nchunks = (w.kv_len + 31) >> 5;
  const int tail0 = FUSED ? bv.work[item].tail0 : w.kv_len;
  const int ctail = tail0 >> 5;  // first chunk read from the LDS tail
  h8 kf0[2][KS], va0[DT];
  // this wave's chunks: c0, c0 + cstep, ...
  const int c0 = ZS ? (int)blockIdx.z * NW + wave : wave, cstep = ZS ? NW * (int)gridDim.z : NW;
  const bool early = FUSED && c0 < nchunks && c0 < ctail;

  // OP: this head's K-slice of Wo (k-steps h*KS .. h*KS + KS - 1) for the
  // wave's column tiles, issued right behind the prologue's loads (and the
  // first K/V chunk), so the KV update, key loop and merge hide its latency
  constexpr int OT = OP ? 8 : 1;
  h8 wo_f[OT][KS];
  const int o_tiles = OP ? opa.N >> 4 : 0;
  auto load_wo = [&]() {
    if constexpr (OP) {
#pragma unroll
      for (int j = 0; j < OT; ++j) {
        const int t = (wave + j * NW) * (int)gridDim.z + (int)blockIdx.z;  // (column split)
        if (t < o_tiles) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            wo_f[j][ks] = *reinterpret_cast<const h8 *>(opa.wo + (size_t)t * opa.wts +
                                                        (size_t)(h * KS + ks) * opa.wks + lane * 8);
        }
      }
    }
  };

  // FUSED: this item's rotated queries stay in LDS (rows padded by 16 B)
  __shared__ __attribute__((aligned(16))) uint16_t sQ[FUSED ? NQK : 1][D + 8];
  __shared__ int4 sMrec[FUSED ? NQK : 1];
  __shared__ int sSlotV[FUSED ? NQK : 1];
  __shared__ uint64_t sMvis[FUSED ? NQK : 1];
  if (FUSED) {
    int *sSlot = sSlotV;
    const WorkDev *wdp = &bv.work[item];
    // the queries' visibility records go out with the prologue's loads and
    // reach the key loop through LDS (a load there was one more round trip)
    int4 mrec;
    uint64_t mvis;
    constexpr int NT = 64 * NW;
    constexpr int D8 = D / 8;
    // cached contents of the tail's first `told` (< 32) slots, which this
    // step does not write, 16-B pieces: K rows, then V^T row segments (the
    // V^T pieces cover the whole first chunk; the written slots among them
    // are overwritten in LDS after the barrier below)
    constexpr int TK = (32 * D8 + NT - 1) / NT, TV = (D * 4 + NT - 1) / NT;
    const int told = wdp->told;
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));  // (arrays of the struct uint4 go to scratch)
    v4 tk[TK], tv[TV];
    // the request's commits (16-B pieces of the staging K and V rows)
    constexpr int CP = (kItemCommits * 2 * D8 + NT - 1) / NT;
    const int ncm = kv.C > 0 ? wdp->ncommit : 0;
    // commit sources through the scalar cache, with the work item: the
    // staging loads then wait on no vector load (one round trip, not two)
    // (readfirstlane keeps them scalar: a select over the loaded words was
    // folded into a per-lane load that the staging loads then waited for)
    const uint32_t *cs32 = reinterpret_cast<const uint32_t *>(wdp->cm_src);
    uint32_t csw[kItemCommits / 2];
#pragma unroll
    for (int jj = 0; jj < kItemCommits / 2; ++jj) csw[jj] = __builtin_amdgcn_readfirstlane(cs32[jj]);
    int csrc[CP];  // this thread's commit pieces: source staging rows
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const int j = min(((int)threadIdx.x + i * NT) / (2 * D8), kItemCommits - 1);
      uint32_t wd = csw[0];
#pragma unroll
      for (int jj = 1; jj < kItemCommits / 2; ++jj) wd = (j >> 1) == jj ? csw[jj] : wd;
      csrc[i] = (int)(int16_t)((j & 1) ? (wd >> 16) : (wd & 0xffffu));
    }
    v4 cmv[CP];
    kv_update_item<D, NQK, NT, PSRC>(
        bv, wdp, h, heads, slots, kv.T, kv.qkv, kv.part, kv.pS, kv.pNP, kv.rope, kv.max_rope_pos,
        qbuf, kc, kv.stage_wr, nullptr, sSlot, sQ, sKt, sVt, tail0,
        [&] {  // after the KV update's own loads: commits, tail, first chunk
#pragma unroll
          for (int i = 0; i < CP; ++i) {
            const int e = threadIdx.x + i * NT, j = e / (2 * D8), r = e % (2 * D8);
            if (j < ncm) {
              const int src = csrc[i];
              cmv[i] = *reinterpret_cast<const v4 *>(
                  kv.stage_rd + (size_t)src * 2 * Hl + (r >= D8 ? Hl : 0) + h * D + (r % D8) * 8);
            }
          }
#pragma unroll
          for (int i = 0; i < TK; ++i) {
            const int e = threadIdx.x + i * NT, row = e / D8;
            if (row < told)
              tk[i] = *reinterpret_cast<const v4 *>(kbase + (size_t)(tail0 + row) * D + (e % D8) * 8);
          }
#pragma unroll
          for (int i = 0; i < TV; ++i) {
            const int e = threadIdx.x + i * NT, dd = e / 4, s8 = (e % 4) * 8;
            if (dd < D && s8 < told)
              tv[i] = *reinterpret_cast<const v4 *>(vbase + (size_t)dd * slots + tail0 + s8);
          }
          if ((int)threadIdx.x < NQK) {
            const ffmi_token_info *ti = &bv.tokens[w.q_start + min((int)threadIdx.x, max(w.q_count - 1, 0))];
            mrec = make_int4(ti->prefix_len, ti->tree_base, ti->tree_len, 0);
            mvis = ti->tree_vis;
          }
          // (issued last: the waits below for the loads above leave it in flight)
          if (early) load_chunk(c0, kf0, va0);
          load_wo();
        },
        [&] {  // loads are back: the old tail to LDS, then the commits
          stamp(10);
          if ((int)threadIdx.x < NQK) sMrec[threadIdx.x] = mrec, sMvis[threadIdx.x] = mvis;
#pragma unroll
          for (int i = 0; i < TK; ++i) {
            const int e = threadIdx.x + i * NT, row = e / D8;
            if (row < told) *reinterpret_cast<v4 *>(&sKt[row][(e % D8) * 8]) = tk[i];
          }
#pragma unroll
          for (int i = 0; i < TV; ++i) {
            const int e = threadIdx.x + i * NT, dd = e / 4, s8 = (e % 4) * 8;
            if (dd < D && s8 < told) {
              uint2 *dst = reinterpret_cast<uint2 *>(&sVt[dd][s8]);
              dst[0] = make_uint2(tv[i].x, tv[i].y);
              dst[1] = make_uint2(tv[i].z, tv[i].w);
            }
          }
          stamp(11);
          // keys past kv_len in the last chunk are masked, but P.V still
          // multiplies their V by 0: zero them (as the cache's never-written
          // slots are); a stored slot among them is written after the barrier
          for (int e = threadIdx.x; e < D * 32; e += NT) {
            const int dd = e >> 5, sl = w.kv_len - tail0 + (e & 31);
            if (sl < (nchunks - ctail) * 32) sVt[dd][sl] = 0;
          }
          __syncthreads();
          // commits (tree_inc...cu:335-396): staging row -> depth slot, in
          // HBM and in the tail (their slots differ from this step's stores:
          // a coinciding commit was applied by its own launch, kv.C == 0)
#pragma unroll
          for (int i = 0; i < CP; ++i) {
            const int e = threadIdx.x + i * NT, j = e / (2 * D8), r = e % (2 * D8);
            if (j >= ncm) continue;
            const int dep = wdp->cm_depth[j], i8 = (r % D8) * 8;
            if (dep < 0 || dep >= slots) continue;
            const int ts = dep - tail0;
            if (r < D8) {
              *reinterpret_cast<v4 *>(kc + (((size_t)w.req * heads + h) * slots + dep) * D + i8) =
                  cmv[i];
              *reinterpret_cast<v4 *>(&sKt[ts][i8]) = cmv[i];
            } else {
              uint16_t *vt = vc + (((size_t)w.req * heads + h) * D + i8) * slots + dep;
              const uint32_t vw[4] = {cmv[i].x, cmv[i].y, cmv[i].z, cmv[i].w};
#pragma unroll
              for (int jj = 0; jj < 8; ++jj) {
                const uint16_t v = (uint16_t)(vw[jj >> 1] >> (16 * (jj & 1)));
                vt[(size_t)jj * slots] = v;
                sVt[i8 + jj][ts] = v;
              }
            }
          }
          stamp(6);
        });
    stamp(7);
    __syncthreads();
    stamp(8);
    stamp(9);
  }

  stamp(1);
  bool qvalid[QT];
  int pre[QT], tb[QT], tlen[QT];
  uint64_t tv[QT];
  h8 qf[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int q = qbase + qt * 16 + qi;
    qvalid[qt] = q < w.q_count;
    if (FUSED) {
      const int4 mr = sMrec[qvalid[qt] ? q : 0];
      pre[qt] = mr.x, tb[qt] = mr.y, tlen[qt] = mr.z, tv[qt] = sMvis[qvalid[qt] ? q : 0];
    } else {
      const ffmi_token_info ti = bv.tokens[w.q_start + (qvalid[qt] ? q : 0)];
      pre[qt] = ti.prefix_len, tb[qt] = ti.tree_base, tlen[qt] = ti.tree_len, tv[qt] = ti.tree_vis;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qt][ks] = !qvalid[qt] ? h8{0, 0, 0, 0, 0, 0, 0, 0}
                   : FUSED ? *reinterpret_cast<const h8 *>(&sQ[q][32 * ks + 8 * g])
                           : *reinterpret_cast<const h8 *>(
                                 qbuf + (size_t)(w.q_start + q) * Hl + h * D + 32 * ks + 8 * g);
  }

  const float NEG = -INFINITY;
  int seen[QT];  // slots below it are visible to the lane's query
  float m_run[QT], l_run[QT];
  f4 o[QT][DT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = NEG, l_run[qt] = 0.f;
    seen[qt] = qvalid[qt] ? min(pre[qt], w.kv_len) : INT32_MAX;
#pragma unroll
    for (int t = 0; t < DT; ++t) o[qt][t] = f4{0.f, 0.f, 0.f, 0.f};
  }

  auto compute_chunk = [&](int base, const h8 (&kf)[2][KS], const h8 (&va)[DT]) {
    attn_chunk<D, QT>(base, g, kf, va, qf, qvalid, seen, pre, tb, tlen, tv, w.kv_len, scale, m_run, l_run, o);
  };
  // A wave's chunks with the next one's loads in flight while it computes: keys
  // and values with one query tile, the keys with two (two tiles' outputs leave
  // no registers for a second set of values; those are asked for before the
  // next scores).  Waiting for each chunk in turn, at about 1500 keys: 42.6 us
  // for one query of each of 4 requests (16 heads, d = 128), now 29.8; 69 us for
  // a step's 33 prompt items, now 60.
  // FUSED: chunks from ctail on come from the LDS tail
  auto load_chunk_lds = [&](int lc, h8 (&kf)[2][KS], h8 (&va)[DT]) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const uint16_t *krow = &sKt[lc * 32 + krow0 + 4 * sub][8 * g];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[sub][ks] = *reinterpret_cast<const h8 *>(krow + 32 * ks);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      va[t] = *reinterpret_cast<const h8 *>(&sVt[t * 16 + (lane & 15)][lc * 32 + 8 * g]);
    }
  };
  stamp(2);
  const int cend = FUSED ? min(ctail, nchunks) : nchunks;
  int c = c0;
  if (!FUSED && c < cend) load_chunk(c, kf0, va0);
  for (; c < cend; c += cstep) {
    const bool more = c + cstep < cend;
    h8 kf1[2][KS], va1[QT == 1 ? DT : 1];
    if (more) load_keys(c + cstep, kf1);
    if constexpr (QT == 1) {
      if (more) load_values(c + cstep, va1);
      compute_chunk(c * 32, kf0, va0);
#pragma unroll
      for (int t = 0; t < DT; ++t) va0[t] = va1[t];
    } else {
      compute_chunk(c * 32, kf0, va0);
      if (more) load_values(c + cstep, va0);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf0[0][ks] = kf1[0][ks], kf0[1][ks] = kf1[1][ks];
  }
  if constexpr (FUSED)
    for (; c < nchunks; c += cstep) {
      h8 kf[2][KS], va[DT];
      load_chunk_lds(c - ctail, kf, va);
      compute_chunk(c * 32, kf, va);
    }

  stamp(3);
  if (FUSED) {
    // V^T of this step's tokens to HBM from the tail, by each wave once its
    // key loop is done (not waited for)
    uint16_t *vt = vc + ((size_t)w.req * heads + h) * D * slots;
    for (int e = threadIdx.x; e < D * NQK; e += blockDim.x) {
      const int dd = e / NQK, tt = e % NQK;
      if (tt >= w.q_count) continue;
      const int sl = sSlotV[tt];
      if (sl >= 0) vt[(size_t)dd * slots + sl] = sVt[dd][sl - tail0];
    }
    __syncthreads();  // the merge buffer reuses the tail's LDS
  }
  // per-query partial sum over the 4 lane groups (same m_run in all four)
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float l = l_run[qt];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) {
      sm_m[wave][qt * 16 + qi] = m_run[qt];
      sm_l[wave][qt * 16 + qi] = l;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) sm_o[wave][qt][t][r][lane] = o[qt][t][r];
  }
  __syncthreads();
  stamp(4);

  // merge: wave w finalizes d-tiles t = w, w+NW, ... of every query tile
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int ql = qt * 16 + qi, q = qbase + ql;  // in the workgroup / in the item
    float M = NEG;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, sm_m[ww][ql]);
    float f[NW], L = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const float mw = sm_m[ww][ql];
      f[ww] = (mw == NEG) ? 0.f : __expf(mw - M);
      L += f[ww] * sm_l[ww][ql];
    }
    if constexpr (ZS) {
      // the partial outputs past every cache, then the count; the last one merges
      const int pair = w.req * heads + h, Z = (int)gridDim.z;
      float *mine = kv.zpart + ((size_t)pair * kv.zmax + blockIdx.z) * (D + 2);
      if (wave < DT && qi == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float acc = 0.f;
#pragma unroll
          for (int ww = 0; ww < NW; ++ww) acc += f[ww] * sm_o[ww][qt][wave][r][lane];
          __hip_atomic_store(mine + wave * 16 + 4 * g + r, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (threadIdx.x == 0) {
        __hip_atomic_store(mine + D, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mine + D + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        const unsigned before =
            __hip_atomic_fetch_add(kv.zcount + pair, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sMrec[0].w = before + 1 == (unsigned)Z;
        if (before + 1 == (unsigned)Z)
          __hip_atomic_store(kv.zcount + pair, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      const int dd = (int)threadIdx.x * 2;
      if (!sMrec[0].w || dd >= D || w.q_count == 0) return;
      const float *all = kv.zpart + (size_t)pair * kv.zmax * (D + 2);
      float zm[kMaxKvSplit], zl[kMaxKvSplit], za[kMaxKvSplit], zb[kMaxKvSplit];
#pragma unroll
      for (int z = 0; z < kMaxKvSplit; ++z) {  // (all in flight; past Z the last one again)
        const float *q = all + (size_t)min(z, Z - 1) * (D + 2);
        zm[z] = __hip_atomic_load(q + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        zl[z] = __hip_atomic_load(q + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        za[z] = __hip_atomic_load(q + dd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        zb[z] = __hip_atomic_load(q + dd + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float zM = NEG, zL = 0.f, oa = 0.f, ob = 0.f;
#pragma unroll
      for (int z = 0; z < kMaxKvSplit; ++z) zM = fmaxf(zM, zm[z]);
#pragma unroll
      for (int z = 0; z < kMaxKvSplit; ++z) {
        const float e = z >= Z || zm[z] == NEG ? 0.f : __expf(zm[z] - zM);
        zL += e * zl[z], oa += e * za[z], ob += e * zb[z];
      }
      const float zinv = 1.0f / (zL + 1e-6f);
      uint16_t *dst = out_packed ? out + act_packed_off(w.q_start, h * D + dd, Hl)
                                 : out + (size_t)w.q_start * Hl + h * D + dd;
      *reinterpret_cast<uint32_t *>(dst) = f2h(oa * zinv) | ((uint32_t)f2h(ob * zinv) << 16);
      return;
    }
    const float inv = 1.0f / (L + 1e-6f);
    if (!qvalid[qt]) continue;
    const int orow_m = w.q_start + q;
    uint16_t *orow = out + (size_t)orow_m * Hl + h * D;
    for (int t = wave; t < DT; t += NW) {
      uint16_t r4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) acc += f[ww] * sm_o[ww][qt][t][r][lane];
        r4[r] = f2h(acc * inv);
      }
      uint2 pk;
      pk.x = r4[0] | ((uint32_t)r4[1] << 16);
      pk.y = r4[2] | ((uint32_t)r4[3] << 16);
      uint16_t *dst = out_packed ? out + act_packed_off(orow_m, h * D + t * 16 + 4 * g, Hl)
                                 : orow + t * 16 + 4 * g;
      *reinterpret_cast<uint2 *>(dst) = pk;
      // OP: the rounded row also to LDS (the queries' tile is free by now)
      if (OP) *reinterpret_cast<uint2 *>(&sQ[q][t * 16 + 4 * g]) = pk;
    }
  }
  if constexpr (OP) {
    // slab[head][token][n] = sum_d out[token][head*d + d] * Wo[n][head*d + d]:
    // lane (qi, g) ends with n = 16 t + 4 g + r of query qi.  Rows of queries
    // past q_count hold stale LDS; their columns are computed, never stored.
    __syncthreads();
    h8 xb[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xb[ks] = *reinterpret_cast<const h8 *>(&sQ[qi][32 * ks + 8 * g]);
    const bool qv = qi < w.q_count;
    float *srow = opa.slab + ((size_t)h * kv.T + w.q_start + qi) * opa.N + 4 * g;
#pragma unroll
    for (int j = 0; j < OT; ++j) {
      const int t = (wave + j * NW) * (int)gridDim.z + (int)blockIdx.z;
      if (t < o_tiles) {
        f4 c = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(wo_f[j][ks], xb[ks], c, 0, 0, 0);
        if (qv) *reinterpret_cast<f4 *>(srow + t * 16) = c;
      }
    }
  }
  if (ST && stp) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    stamp(5);
  }
}

// Prompt items (several work items of a request): one workgroup per (two
// consecutive items of a request, head), its keys through LDS in stages of 128,
// the next stage on its way while one is computed.  Waves 0-3 attend the first
// item's 32 queries, 4-7 the second's, each a quarter of a stage's keys.
// Loading its own chunks a wave's lanes go to 16 rows of K at a time (the MFMA
// operand), which the L1 serves one 16-byte access after another; here a wave
// copies whole rows (16-byte pieces exchanged in a row by its number, so that the
// operand reads hit different banks) and both items use them.  33 items x 16
// heads, d = 128, at about 1500 keys: 47 us one by one, 35 here, about 2.2 us per
// stage on a CU, of which the LDS reads, the MFMA and the softmax are about half;
// the rest waits for the next stage (two of them fill the LDS).
constexpr int kBlockKeys = 128;
template <int D>
__global__ __launch_bounds__(512, 1) void attention_block_kernel(
    const char *__restrict__ blob, const uint16_t *__restrict__ qbuf, const uint16_t *__restrict__ kc,
    const uint16_t *__restrict__ vc, uint16_t *__restrict__ out, int heads, int slots, float scale,
    int out_packed) {
  constexpr int KS = D / 32, DT = D / 16, QT = 2, D8 = D / 8;
  constexpr int NB = kBlockKeys * D * 2 / 1024;  // 1-KiB pieces of a stage's K, and of its V^T
  constexpr int PW = NB / 8;                     // of each, a wave's
  __shared__ h8 lds[2][2 * NB * 64];
  __shared__ float sm_m[8][32], sm_l[8][32];
  const int lane = threadIdx.x & 63, qi = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qg = wave >> 2, kg = wave & 3;
  int at, h;
  attn_place(at, h, (int)gridDim.x, (int)gridDim.y);
  const BatchView bv = batch_view(blob);
  // (the later, longer items of a request first)
  const int block = bv.work[(int)gridDim.x - 1 - at].block;
  const int first = block >> 1, count = 1 + (block & 1);
  const ffmi_attn_work w = bv.work[first + min(qg, count - 1)].w;
  const int nchunks = (max(bv.work[first].w.kv_len, bv.work[first + count - 1].w.kv_len) + 31) >> 5;
  const int nmine = qg < count ? (w.kv_len + 31) >> 5 : 0;
  const int Hl = heads * D;
  const uint16_t *kbase = kc + ((size_t)w.req * heads + h) * slots * D;
  const uint16_t *vbase = vc + ((size_t)w.req * heads + h) * D * slots;

  bool qvalid[QT];
  int pre[QT], tb[QT], tlen[QT], seen[QT];
  uint64_t tv[QT];
  h8 qf[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int q = qt * 16 + qi;
    qvalid[qt] = qg < count && q < w.q_count;
    // (columns past q_count: the first query again, never stored)
    const int t = w.q_start + (qvalid[qt] ? q : 0);
    const ffmi_token_info ti = bv.tokens[t];
    pre[qt] = ti.prefix_len, tb[qt] = ti.tree_base, tlen[qt] = ti.tree_len, tv[qt] = ti.tree_vis;
    seen[qt] = qvalid[qt] ? min(pre[qt], w.kv_len) : INT32_MAX;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qt][ks] = *reinterpret_cast<const h8 *>(qbuf + (size_t)t * Hl + h * D + 32 * ks + 8 * g);
  }
  // stage st to buffer buf (chunks past the last one: the last one again, unread)
  auto copy = [&](int st, int buf) {
    auto put = [&](const uint16_t *src, int piece) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                       (__attribute__((address_space(3))) void *)&lds[buf][piece * 64],
                                       16, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int row = (wave * PW + i) * (64 / D8) + lane / D8;
      const int piece = lane % D8 ^ (((row & 3) | (row >> 3 & 3) << 2) & (D8 - 1));
      const int key = min(4 * st + (row >> 5), nchunks - 1) * 32 + (row & 31);
      put(kbase + (size_t)key * D + piece * 8, wave * PW + i);
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int row = (wave * PW + i) * 4 + (lane >> 4), piece = (lane ^ row) & 15;
      const int key = min(4 * st + (piece >> 2), nchunks - 1) * 32 + (piece & 3) * 8;
      put(vbase + (size_t)row * slots + key, NB + wave * PW + i);
    }
  };
  const float NEG = -INFINITY;
  float m_run[QT], l_run[QT];
  f4 o[QT][DT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = NEG, l_run[qt] = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t) o[qt][t] = f4{0.f, 0.f, 0.f, 0.f};
  }
  const int krow = kg * 32 + 8 * (qi >> 2) + (qi & 3);  // (+ 4 sub: attention_kernel's order)
  const int stages = (nchunks + 3) >> 2;
  if (stages > 0) copy(0, 0);
  if (stages > 1) copy(1, 1);
  for (int st = 0; st < stages; ++st) {
    // this stage's copies are there (the next one's 2 PW stay in flight)
    if (st + 1 < stages) __builtin_amdgcn_s_waitcnt((2 * PW & 15) | 0x0f70);
    else __builtin_amdgcn_s_waitcnt(0x0f70);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (4 * st + kg < nmine) {
      const h8 *sk = lds[st & 1], *sv = sk + NB * 64;
      h8 kf[2][KS], va[DT];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          kf[sub][ks] = sk[(krow + 4 * sub) * D8 + ((4 * ks + g) ^ (qi & (D8 - 1)))];
#pragma unroll
      for (int t = 0; t < DT; ++t) va[t] = sv[(t * 16 + qi) * 16 + ((4 * kg + g) ^ qi)];
      attn_chunk<D, QT>((4 * st + kg) * 32, g, kf, va, qf, qvalid, seen, pre, tb, tlen, tv, w.kv_len, scale,
                        m_run, l_run, o);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads are back
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (st + 2 < stages) copy(st + 2, st & 1);
  }
  // merge of the four quarters, as attention_kernel's of its waves
  auto sm_o = reinterpret_cast<float(*)[QT][DT][4][64]>(&lds[0][0]);
  static_assert(sizeof(lds) >= 8 * QT * DT * 4 * 64 * 4, "merge buffer");
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float l = l_run[qt];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) sm_m[wave][qt * 16 + qi] = m_run[qt], sm_l[wave][qt * 16 + qi] = l;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) sm_o[wave][qt][t][r][lane] = o[qt][t][r];
  }
  __syncthreads();
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int q = qt * 16 + qi;
    float M = NEG, f[4], L = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) M = fmaxf(M, sm_m[qg * 4 + k][q]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float mw = sm_m[qg * 4 + k][q];
      f[k] = (mw == NEG) ? 0.f : __expf(mw - M);
      L += f[k] * sm_l[qg * 4 + k][q];
    }
    const float inv = 1.0f / (L + 1e-6f);
    if (!qvalid[qt]) continue;
    const int row = w.q_start + q;
    for (int t = kg; t < DT; t += 4) {
      uint16_t r4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float acc = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc += f[k] * sm_o[qg * 4 + k][qt][t][r][lane];
        r4[r] = f2h(acc * inv);
      }
      const int col = h * D + t * 16 + 4 * g;
      st_h4(out_packed ? out + act_packed_off(row, col, Hl) : out + (size_t)row * Hl + col, r4[0], r4[1], r4[2],
            r4[3]);
    }
  }
}

// FFMI_ATTN_BLOCK=0: prompt items one by one (A/B, tests)
static bool attn_block() {
  const char *e = getenv("FFMI_ATTN_BLOCK");
  return !e || atoi(e);
}

static int attn_cus() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      cus = 256;
  }
  return cus;
}
// a doubled grid still fits one wave of the device's CUs
static bool attn_split_fits(int wgs) { return 2 * wgs <= attn_cus(); }

// Workgroups that share an item's keys in a step of one query per request: as
// many as the chip has room for, at least a chunk of 32 keys per wave each (4
// requests x 16 heads, d = 128, about 1500 keys: 29.8 us with one each, 16.3
// with four), where that saves more than the merge's 1.3-2 us.  A round of 8 chunks
// is 3.3 us at d = 128, 1.5 at 64 and 0.5 at 32, so from how many chunks on it pays
// depends on d (one workgroup each / shared, 4 requests x 16 heads: d = 128, 300 keys 11.4 /
// 11.2, 450 11.7 / 10.4; d = 64, 300 keys 8.1 / 8.7, 513 8.6 / 8.5, 700 10.4 / 8.9; d = 32,
// 513 keys 6.2 / 7.7, 1025 7.2 / 8.1).  With a workgroup on every CU there is nothing to gain.
// FFMI_ATTN_KVSPLIT=0: one (A/B, tests).
int attn_kv_split(int W, int heads, int d, int max_q, int max_kv) {
  const int chunks = (max_kv + 31) / 32;
  if (max_q != 1 || W <= 0 || chunks <= (d >= 128 ? 8 : d >= 64 ? 16 : 40)) return 1;
  const int room = std::min(attn_cus(), kKvSplitWgs) / (W * heads);
  const int Z = std::max(1, std::min(std::min(room, (chunks + 7) / 8), kMaxKvSplit));
  const char *e = Z > 1 ? getenv("FFMI_ATTN_KVSPLIT") : nullptr;
  return e && !atoi(e) ? 1 : Z;
}

// Query split (attention_kernel QS == 2) of a fused launch with more than 16
// queries per item: when the (item, head) grid leaves half the CUs idle
// (TP >= 2 verify steps).  FFMI_ATTN_QSPLIT: 0 off, 1 auto (default), 2
// always (tests; read at every launch, so a test can switch it).
static bool attn_qsplit(int wgs) {
  const char *e = getenv("FFMI_ATTN_QSPLIT");
  const int mode = e ? atoi(e) : 1;
  return mode == 2 || (mode == 1 && attn_split_fits(wgs));
}

static bool attn_osplit(int wgs) {
  const char *e = getenv("FFMI_ATTN_OSPLIT");
  const int mode = e ? atoi(e) : 1;
  return mode == 2 || (mode == 1 && attn_split_fits(wgs));
}

template <int D>
static hipError_t launch_attention_d(const char *blob, int W, int max_q, uint16_t *qbuf,
                                     uint16_t *kc, uint16_t *vc, uint16_t *out, int heads,
                                     int slots, float scale, hipStream_t s, int op, bool fused,
                                     const KvUpdateArgs &kv, int Z, int blocks) {
  const dim3 grid(W, heads);
#define FFMI_ATT(QT, FU)                                                                      \
  do {                                                                                          \
    if (!FU)                                                                                    \
      hipLaunchKernelGGL((attention_kernel<D, QT, 8, false>), grid, dim3(512), 0, s, blob, qbuf, \
                         kc, vc, out, heads, slots, scale, op, kv, OprojArgs());                             \
    else if (kv.part)                                                                           \
      hipLaunchKernelGGL((attention_kernel<D, QT, 8, true, false, 1>), grid, dim3(512), 0, s,    \
                         blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());                 \
    else                                                                                        \
      hipLaunchKernelGGL((attention_kernel<D, QT, 8, true, false, 0>), grid, dim3(512), 0, s,    \
                         blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());                 \
  } while (0)
  // diagnostics build: FFMI_ATTN_STAMP=1 stamps the d = 128 (LLM) launches,
  // FFMI_ATTN_STAMP=64 the d = 64 (68M SSM) ones
  static const int stamp_d = getenv("FFMI_ATTN_STAMP") && atoi(getenv("FFMI_ATTN_STAMP")) == 64 ? 64 : 128;
  if (kv.stamps && D == stamp_d) {
#define FFMI_ATT_ST(QT)                                                                         \
  do {                                                                                          \
    if (fused)                                                                                  \
      hipLaunchKernelGGL((attention_kernel<D, QT, 8, true, true>), grid, dim3(512), 0, s, blob,  \
                         qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());                       \
    else                                                                                        \
      hipLaunchKernelGGL((attention_kernel<D, QT, 8, false, true>), grid, dim3(512), 0, s, blob, \
                         qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());                       \
  } while (0)
    if (max_q > 16) FFMI_ATT_ST(2);
    else FFMI_ATT_ST(1);
#undef FFMI_ATT_ST
    return hipGetLastError();
  }
  if (fused && Z > 1) {
    const dim3 gridz(W, heads, Z);
    if (kv.part)
      hipLaunchKernelGGL((attention_kernel<D, 1, 8, true, false, 1, false, 1, true>), gridz, dim3(512), 0,
                         s, blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
    else
      hipLaunchKernelGGL((attention_kernel<D, 1, 8, true, false, 0, false, 1, true>), gridz, dim3(512), 0,
                         s, blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
    return hipGetLastError();
  }
  if (max_q > 16 && fused && attn_qsplit(W * heads)) {
    const dim3 grid2(W, heads, 2);
    if (kv.part)
      hipLaunchKernelGGL((attention_kernel<D, 1, 8, true, false, 1, false, 2>), grid2, dim3(512), 0,
                         s, blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
    else
      hipLaunchKernelGGL((attention_kernel<D, 1, 8, true, false, 0, false, 2>), grid2, dim3(512), 0,
                         s, blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
    return hipGetLastError();
  }
  // more workgroups than CUs: items of several tokens blocks of two (up to a CU
  // each, the waves of one item in its own workgroup: 8 items x 32 heads 8.4 us,
  // in blocks 9.4); single queries four waves each, two workgroups to a CU (9 items
  // x 32 heads at about 260 keys: 17.7 us with eight waves, two rounds, now 15.7;
  // eight are the faster ones while a CU each is enough)
  if (W * heads > attn_cus() && !kv.stamps) {
    if constexpr (D >= 64)
      if (blocks > 0 && max_q > 16 && !fused && attn_block()) {
        hipLaunchKernelGGL(attention_block_kernel<D>, dim3(blocks, heads), dim3(512), 0, s, blob, qbuf, kc,
                           vc, out, heads, slots, scale, op);
        return hipGetLastError();
      }
    if (max_q == 1 && fused) {
      if (kv.part)
        hipLaunchKernelGGL((attention_kernel<D, 1, 4, true, false, 1>), grid, dim3(256), 0, s, blob, qbuf,
                           kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
      else
        hipLaunchKernelGGL((attention_kernel<D, 1, 4, true, false, 0>), grid, dim3(256), 0, s, blob, qbuf,
                           kc, vc, out, heads, slots, scale, op, kv, OprojArgs());
      return hipGetLastError();
    }
  }
  if (max_q <= 16) {
    if (fused) FFMI_ATT(1, true);
    else FFMI_ATT(1, false);
  } else {
    if (fused) FFMI_ATT(2, true);
    else FFMI_ATT(2, false);
  }
#undef FFMI_ATT
  return hipGetLastError();
}

// FFMI_ATTN_STAMP=1: d = 128 launches record a per-wave timeline
// {start, after prologue, before k-loop, after k-loop, after merge barrier,
// end, [fused] after commits, after KV update, after its barrier, after the
// V^T stores, HW_ID, chunks} (100 MHz realtime) for ffmi_debug_attn_stamps.
static long long *g_attn_stamps = nullptr;
static long g_attn_stamp_waves = 0;
static bool g_attn_stamp_gate = true;
// the model closes the gate for every launch but the one its markers bracket
void attn_stamp_gate(bool open) { g_attn_stamp_gate = open; }
static long long *attn_stamp_buf(int wgs) {
  static const bool on = getenv("FFMI_ATTN_STAMP") != nullptr;
  if (!on) return nullptr;
  // (allocated on the first launch, gate open or not: a later first use may
  // sit inside a graph capture, where hipMalloc fails)
  if (!g_attn_stamps && hipMalloc(&g_attn_stamps, (size_t)8 << 20) != hipSuccess) return nullptr;
  if (!g_attn_stamp_gate) return nullptr;
  g_attn_stamp_waves = std::min<long>((long)wgs * 8, ((long)8 << 20) / 96);
  return g_attn_stamps;
}

// FFMI_MARKERS=1 diagnostics: a one-wave kernel that records the 100 MHz
// realtime clock (the attention stamps' clock) into slot i when it starts,
// enqueued between the kernels of the model's last layer: with the wave
// stamps it splits a launch's duration into boundary and in-kernel time.
__global__ void marker_kernel(long long *buf, int i) {
  if (threadIdx.x == 0) buf[i] = __builtin_amdgcn_s_memrealtime();
}
static long long *g_markers = nullptr;
hipError_t launch_marker(int i, hipStream_t s) {
  if (i < 0 || i >= 64) return hipErrorInvalidValue;
  if (!g_markers && hipMalloc(&g_markers, 64 * sizeof(long long)) != hipSuccess)
    return hipErrorOutOfMemory;
  hipLaunchKernelGGL(marker_kernel, dim3(1), dim3(64), 0, s, g_markers, i);
  return hipGetLastError();
}
long debug_markers(long long *dst, long n) {
  if (!g_markers || n <= 0) return 0;
  n = std::min<long>(n, 64);
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (hipMemcpy(dst, g_markers, (size_t)n * sizeof(long long), hipMemcpyDeviceToHost) != hipSuccess)
    return -1;
  return n;
}

long attn_debug_stamps(long long *dst, long max_waves) {
  if (!g_attn_stamps || max_waves <= 0) return 0;
  const long n = std::min(max_waves, g_attn_stamp_waves);
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (hipMemcpy(dst, g_attn_stamps, (size_t)n * 96, hipMemcpyDeviceToHost) != hipSuccess) return -1;
  return n;
}

// fused == false: the KV of this step must already be in the cache
// (launch_kv_update); fused == true: one workgroup per request (checked by the
// caller) does commits + KV update + attention.
hipError_t launch_attention(const char *blob, int W, int max_q, uint16_t *qbuf, uint16_t *kc,
                            uint16_t *vc, uint16_t *out, int heads, int d, int slots, float scale,
                            hipStream_t s, bool out_packed, bool fused, int T, int C,
                            const uint16_t *qkv, Partials qkvp, uint16_t *stage_wr,
                            const uint16_t *stage_rd, const float *rope, int max_rope_pos,
                            const OprojArgs *opa, int Z, float *zscratch, int requests, int blocks) {
  if (W <= 0) return hipSuccess;
  if (out_packed && (heads * d) % 32) return hipErrorInvalidValue;
  if (max_q > FFMI_ATTN_QTILE) return hipErrorInvalidValue;
  const int zmax = kv_split_most(heads);
  const KvUpdateArgs kv{T,        C,        qkv,  qkvp.S > 0 ? qkvp.p : nullptr,
                        qkvp.S,   qkvp.NP,  stage_wr, stage_rd,
                        rope,     max_rope_pos, attn_stamp_buf(W * heads),
                        zscratch ? zscratch + (size_t)requests * heads : nullptr, (unsigned *)zscratch, zmax};
  if (Z > 1 && (!fused || !zscratch || max_q != 1 || Z > zmax))
    return hipErrorInvalidValue;
  const int op = out_packed ? 1 : 0;
  if (opa) {  // output projection folded in (the caller checked fused, d, max_q, N)
    if (!fused || d != 64 || max_q > 16 || opa->N % 16 || opa->N > 16 * 8 * 8 || T > opa->max_T)
      return hipErrorInvalidValue;
    // output-column split: when the (item, head) grid leaves half the CUs
    // idle (the 68M SSM: 8 x 12 = 96 workgroups), two workgroups per (item,
    // head) each project half of the column tiles; both attend and run the
    // KV update (the same values to the same addresses, as the query split).
    // The projection's weight slice (96 KiB) and MFMAs per workgroup halve:
    // SSM step 102.9 -> 100.4 us over 5 same-box pairs (profiles/r04_attn_osplit_ab.log).
    // FFMI_ATTN_OSPLIT: 0 off, 1 auto (default), 2 always (read per launch).
    const dim3 grid(W, heads, attn_osplit(W * heads) ? 2 : 1);
    if (kv.part)
      hipLaunchKernelGGL((attention_kernel<64, 1, 8, true, false, 1, true>), grid, dim3(512), 0, s,
                         blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, *opa);
    else
      hipLaunchKernelGGL((attention_kernel<64, 1, 8, true, false, 0, true>), grid, dim3(512), 0, s,
                         blob, qbuf, kc, vc, out, heads, slots, scale, op, kv, *opa);
    return hipGetLastError();
  }
  if (d == 128)
    return launch_attention_d<128>(blob, W, max_q, qbuf, kc, vc, out, heads, slots, scale, s, op,
                                   fused, kv, Z, blocks);
  if (d == 64)
    return launch_attention_d<64>(blob, W, max_q, qbuf, kc, vc, out, heads, slots, scale, s, op,
                                  fused, kv, Z, blocks);
  if (d == 32)  // incremental decoding's third head size (inc...cu:911-926)
    return launch_attention_d<32>(blob, W, max_q, qbuf, kc, vc, out, heads, slots, scale, s, op,
                                  fused, kv, Z, blocks);
  return hipErrorInvalidValue;
}

}  // namespace ffmi
