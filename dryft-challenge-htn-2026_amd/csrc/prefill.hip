// Prefill (the prompt pass, engine.py:459-515 with pos = None), gfx950: token-major q/k
// RMSNorm + RoPE + K/V cache write, and causal GQA flash attention over the cache. Both take a
// packed ("varlen") batch: the B prompts' tokens laid end to end, T tokens in all, prompt b
// holding tokens seq_start[b] .. seq_start[b+1] - 1 at positions 0 .. len_b - 1, so a ragged
// batch prefills in one launch per kernel instead of one pass per prompt length.
//
// qkv_prefill_kernel: one workgroup per 16 tokens, a 16-lane group per token taking its heads in
// turn (the raw heads of a batch of 8 requested together); lane j holds dims 4j .. 4j + 3 and
// their rotate-half partners 64 + 4j .. (two 8-byte accesses). Rounding points as the reference's
// (engine.py:107-115, 166-187; fused.py:191-200, 221-257):
//   n = bf16(bf16(x * r) * w), r = 1/sqrt(mean(x^2) + eps)
//   out[d]    = bf16(bf16(n[d] * cos[d]) + bf16(-n[d+64] * sin[d]))        d < 64
//   out[d+64] = bf16(bf16(n[d+64] * cos[d+64]) + bf16(n[d] * sin[d+64]))
// q goes to q_out [T, NH, HD] (token-major), k (normalised, rotated) and v (bit copy) to the
// cache [B, NKV, cap, HD] at (b, kv head, position).
//
// flash_prefill_kernel: one workgroup of 4 waves per (tile of 16 NTT tokens of one prompt, kv
// head). Wave w takes token tile w / (G / HPW) and HPW of the kv head's G query heads, so each K
// and V^T fragment a wave reads from LDS feeds HPW query tiles; the 4 waves stage every 32-key
// block (K and V row-major, V^T read by transposing LDS loads) into LDS once for the whole tile,
// the next block's global loads in flight during the current block. Per block: S^T = K.Q^T on
// MFMA 16x16x32 (A = 16 keys x 32 dims from LDS, B = Q^T held in registers), causal mask key <=
// token position (only on the blocks that reach into the tile), online
// softmax in the log2 domain (scale HD^-0.5 log2 e), P rounded to bf16 (fused.py:335),
// O^T += V^T.P^T; the key order inside each P.V contraction is the one each lane's S^T
// accumulators hold, so P never leaves the lane. A wave skips the blocks past its last token.
// Tiles holding a prompt's last tokens (the longest causal prefixes) are scheduled first.
// flash_prefill_pp_kernel: G = 4 with 32 queries per wave and 64-key blocks staged by LDS-DMA loads.
#include <type_traits>

#include "common.h"

namespace dd {
namespace pf {

constexpr int HD = 128;
constexpr int HALF = 64;
constexpr int KB = 32;                 // keys per block
constexpr int MAXG = 8;                // query heads per kv head
constexpr int KROW = HD + 8;           // LDS K / V row (elements): 272 bytes

// prompt and position of packed token t (seq_start: B + 1 ascending offsets)
__device__ __forceinline__ void locate(const int* __restrict__ seq_start, int B, int t, int& b, int& p) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {                    // last b with seq_start[b] <= t
    const int mid = (lo + hi + 1) >> 1;
    if (seq_start[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  b = lo;
  p = t - seq_start[lo];
}

// One workgroup per 16 tokens: each 16-lane group takes one token's heads in turn, QKV_HPB heads'
// loads in flight together. Lane j of a group holds dims 4j .. 4j + 3 and 64 + 4j .. 64 + 4j + 3
// (two 8-byte accesses), so both rotate-half partners of every dim are in the lane; the head's
// sum of squares is the lane's 8 squares added in order, then reduced over the 16 lanes. The heads are
// split over the grid's second dimension, hpw each: a workgroup's batches of heads are a chain of
// memory round trips, which is all that a short prompt's pass takes (us, graph-timed, 48 heads: 48 /
// 8 / 4 per workgroup): 131 tokens 29.4 / 7.4 / 5.2, 512 30.1 / 8.6 / 7.2, 2,048 32.5 / 16.1 / 13.8,
// 8,192 54.9 / 44.2 / 47.1, 16,223 96.4 / 94.1 / 93.5 (4.3 TB/s; a large copy reaches 4.9).
constexpr int QKV_TPW = 16;            // tokens per workgroup (4 waves x 4 groups)
#ifndef DD_QKV_HPB
#define DD_QKV_HPB 8
#endif
constexpr int QKV_HPB = DD_QKV_HPB;

__device__ __forceinline__ float group16_sum(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ void __launch_bounds__(256)
qkv_prefill_kernel(const bf16* __restrict__ qkv, const bf16* __restrict__ qn,
                   const bf16* __restrict__ kn, const bf16* __restrict__ cos_t,
                   const bf16* __restrict__ sin_t, const int* __restrict__ seq_start, int B, int T,
                   int last_only, bf16* __restrict__ q_out, bf16* __restrict__ kc,
                   bf16* __restrict__ vc, int NH, int NKV, int cap, int rope_rows, float eps,
                   int* __restrict__ err, int hpw) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 15;
  const int t = blockIdx.x * QKV_TPW + wave * 4 + (lane >> 4);   // this group's token
  if (t >= T) return;                                             // whole group
  int b, p;
  locate(seq_start, B, t, b, p);
  const int len = seq_start[b + 1] - seq_start[b];
  if (p < 0 || p >= len || p >= cap || p >= rope_rows) {   // never write outside the cache
    if (j == 0 && blockIdx.y == 0 && err != nullptr) atomicOr(err, 2);
    return;
  }
  // last_only: q of each prompt's last token only, at row b (the last layer's queries)
  const int nheads = NH + 2 * NKV;
  const int h_first = max((int)blockIdx.y * hpw, last_only && p != len - 1 ? NH : 0);
  const int h_end = min(nheads, ((int)blockIdx.y + 1) * hpw);        // this workgroup's heads
  const int d0 = 4 * j, d1 = 64 + 4 * j;
  const size_t cb = (size_t)p * HD;
  const u32x2 c0 = *(const u32x2*)(cos_t + cb + d0), c1 = *(const u32x2*)(cos_t + cb + d1);
  const u32x2 s0 = *(const u32x2*)(sin_t + cb + d0), s1 = *(const u32x2*)(sin_t + cb + d1);
  const u32x2 q0 = *(const u32x2*)(qn + d0), q1 = *(const u32x2*)(qn + d1);
  const u32x2 k0 = *(const u32x2*)(kn + d0), k1 = *(const u32x2*)(kn + d1);
  const float cw[8] = {lo_bf(c0.x), hi_bf(c0.x), lo_bf(c0.y), hi_bf(c0.y),
                       lo_bf(c1.x), hi_bf(c1.x), lo_bf(c1.y), hi_bf(c1.y)};
  const float sw[8] = {lo_bf(s0.x), hi_bf(s0.x), lo_bf(s0.y), hi_bf(s0.y),
                       lo_bf(s1.x), hi_bf(s1.x), lo_bf(s1.y), hi_bf(s1.y)};
  const bf16* row = qkv + (size_t)t * nheads * HD;
  for (int h0 = h_first; h0 < h_end; h0 += QKV_HPB) {
    u32x2 xa[QKV_HPB], xb[QKV_HPB];
#pragma unroll
    for (int i = 0; i < QKV_HPB; ++i) {
      const int h = h0 + i;
      xa[i] = h < h_end ? *(const u32x2*)(row + (size_t)h * HD + d0) : u32x2{0u, 0u};
      xb[i] = h < h_end ? *(const u32x2*)(row + (size_t)h * HD + d1) : u32x2{0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < QKV_HPB; ++i) {
      const int h = h0 + i;
      if (h >= h_end) break;
      if (h >= NH + NKV) {             // v: a straight copy into the cache
        bf16* dst = vc + (((size_t)b * NKV + (h - NH - NKV)) * cap + p) * HD;
        *(u32x2*)(dst + d0) = xa[i];
        *(u32x2*)(dst + d1) = xb[i];
        continue;
      }
      const u32x2 wa = h < NH ? q0 : k0, wb = h < NH ? q1 : k1;
      const float w[8] = {lo_bf(wa.x), hi_bf(wa.x), lo_bf(wa.y), hi_bf(wa.y),
                          lo_bf(wb.x), hi_bf(wb.x), lo_bf(wb.y), hi_bf(wb.y)};
      const float x[8] = {lo_bf(xa[i].x), hi_bf(xa[i].x), lo_bf(xa[i].y), hi_bf(xa[i].y),
                          lo_bf(xb[i].x), hi_bf(xb[i].x), lo_bf(xb[i].y), hi_bf(xb[i].y)};
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) ss += x[k] * x[k];
      ss = group16_sum(ss);
      const float r = rsqrt_ieee(ss / (float)HD + eps);
      float n[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) n[k] = rbf(rbf(x[k] * r) * w[k]);
      // first half: n cos - n[d + 64] sin; second half: n cos + n[d - 64] sin
      float o[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        o[k] = rbf(n[k] * cw[k]) + rbf(-n[k + 4] * sw[k]);
        o[k + 4] = rbf(n[k + 4] * cw[k + 4]) + rbf(n[k] * sw[k + 4]);
      }
      bf16* dst = h < NH ? q_out + ((size_t)(last_only ? b : t) * NH + h) * HD
                         : kc + (((size_t)b * NKV + (h - NH)) * cap + p) * HD;
      *(u32x2*)(dst + d0) = u32x2{pk_bf16(o[0], o[1]), pk_bf16(o[2], o[3])};
      *(u32x2*)(dst + d1) = u32x2{pk_bf16(o[4], o[5]), pk_bf16(o[6], o[7])};
    }
  }
}

struct FlashShared {
  bf16 k[KB][KROW];                    // the block's keys, row-major
  bf16 v[KB][KROW];                    // the block's values, row-major (read transposed)
};

// Tile index -> (prompt, first token position) for tiles of TQ tokens. ntile[b] = ceil(len_b /
// TQ); tiles are numbered prompt by prompt, and workgroup x takes tile (total - 1 - x), so the
// last tiles of the prompts (their longest causal prefixes) go first. last_only: one tile per
// prompt, the one holding its last token.
__device__ __forceinline__ bool tile_of(const int* __restrict__ seq_start, int B, int x, bool last_only,
                                        int TQ, int& b, int& p0) {
  if (last_only) {
    if (x >= B) return false;
    b = x;
    const int len = seq_start[b + 1] - seq_start[b];
    if (len <= 0) return false;
    p0 = ((len - 1) / TQ) * TQ;
    return true;
  }
  int total = 0;
  for (int i = 0; i < B; ++i) total += (seq_start[i + 1] - seq_start[i] + TQ - 1) / TQ;
  const int idx = total - 1 - x;
  if (idx < 0) return false;
  int acc = 0;
  for (int i = 0; i < B; ++i) {
    const int n = (seq_start[i + 1] - seq_start[i] + TQ - 1) / TQ;
    if (idx < acc + n) {
      b = i;
      p0 = (idx - acc) * TQ;
      return true;
    }
    acc += n;
  }
  return false;
}

// q [T, NH, HD] token-major; out [T, NH * HD] (last_only: [B, NH, HD] / [B, NH * HD], row b =
// prompt b's last token). HPW query heads per wave, NTT 16-token tiles per workgroup, with
// NTT * (NH / NKV) / HPW = NWAVE_F waves; MINB workgroups per CU (the register budget).
#ifndef DD_PF_MINB
#define DD_PF_MINB 2
#endif
template <int HPW, int NTT, int NWAVE_F, int MINB>
__global__ void __launch_bounds__(64 * NWAVE_F, MINB)
flash_prefill_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
                     const int* __restrict__ seq_start, int B, int T, bf16* __restrict__ out,
                     int NH, int NKV, int cap, int last_only, float scale_log2) {
  __shared__ FlashShared sh;
  constexpr int TQ = 16 * NTT;
  int b = 0, p0 = 0;
  if (!tile_of(seq_start, B, blockIdx.x, last_only != 0, TQ, b, p0)) return;
  const int G = NH / NKV, kvh = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  const int wpt = G / HPW;                                    // waves per token tile
  const int tt = wave / wpt;                                  // this wave's token tile
  const int head0 = kvh * G + (wave - tt * wpt) * HPW;        // its first query head
  const int s0 = seq_start[b], len = seq_start[b + 1] - s0;
  if (s0 < 0 || len <= 0 || s0 + len > T || len > cap) return;   // inconsistent offsets: no access
  const int pq = p0 + tt * 16 + l16;                          // this lane's query token position
  const bool qok = last_only ? pq == len - 1 : pq < len;
  // the wave's token tile: its last valid position (blocks past it are skipped), and whether
  // any of its lanes holds a query at all
  const int tfirst = p0 + tt * 16;
  const bool wact = last_only ? (len - 1 >= tfirst && len - 1 < tfirst + 16) : tfirst < len;
  const int wlast = min(tfirst + 15, len - 1);
  const int plast = min(p0 + TQ, len) - 1;                    // last query position of the tile
  const int nblk = plast / KB + 1;
  // Q^T operands: lane = token l16, dims kb * 32 + g4 * 8 ..
  u32x4 qreg[HPW][4];
#pragma unroll
  for (int h = 0; h < HPW; ++h)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      qreg[h][kb] = qok ? *(const u32x4*)(q + ((size_t)(last_only ? b : s0 + pq) * NH + head0 + h) * HD +
                                          kb * 32 + g4 * 8)
                        : u32x4{0u, 0u, 0u, 0u};
  f32x4 acc[HPW][8];
  float m_run[HPW], l_run[HPW];
#pragma unroll
  for (int h = 0; h < HPW; ++h) {
    m_run[h] = -INFINITY;
    l_run[h] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[h][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const size_t kvbase = ((size_t)b * NKV + kvh) * cap * HD;
  // staging per block: K and V as 512 16-byte chunks each, 2 of each a thread (chunk c: key
  // c / 16, dims (c % 16) 8 ..), both stored row-major. Buffer loads over this (sequence, kv
  // head)'s cache rows: the per-lane offsets are fixed and the block's key0 goes in the scalar
  // offset; keys past the cache read zeros (they are masked).
  constexpr int CPT = KB * HD / 8 / (64 * NWAVE_F);
  static_assert(CPT * 64 * NWAVE_F * 8 == KB * HD, "whole chunks per thread");
  const rsrc_t kr = make_rsrc(kc + kvbase, (unsigned)((size_t)cap * HD * 2));
  const rsrc_t vr = make_rsrc(vc + kvbase, (unsigned)((size_t)cap * HD * 2));
  unsigned coff[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = (int)threadIdx.x + i * 64 * NWAVE_F;
    coff[i] = (unsigned)((c >> 4) * HD * 2 + (c & 15) * 16);
  }
  u32x4 kst[CPT], vst[CPT];
  auto fetch = [&](int key0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      kst[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, coff[i], (unsigned)key0 * HD * 2, 0);
      vst[i] = __builtin_amdgcn_raw_buffer_load_b128(vr, coff[i], (unsigned)key0 * HD * 2, 0);
    }
  };
  // V^T operand addressing (see lds_read_tr16)
  const int trow = g4 * 4 + (l16 >> 2), tcol = 4 * (l16 & 3);
  // One block: stage it, request the next, then (the wave's keys permitting) add it. MASKED: the
  // causal mask key <= query position; blocks wholly before the tile's first query need none.
  auto block = [&](int blk, auto masked) {
    constexpr bool MASKED = decltype(masked)::value;
    const int key0 = blk * KB;
    __syncthreads();                                          // the previous block is consumed
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = (int)threadIdx.x + i * 64 * NWAVE_F;
      *(u32x4*)&sh.k[c >> 4][(c & 15) * 8] = kst[i];
      *(u32x4*)&sh.v[c >> 4][(c & 15) * 8] = vst[i];
    }
    __syncthreads();
    if (blk + 1 < nblk) fetch(key0 + KB);                     // in flight during this block
    if (!wact || key0 > wlast) return;                        // wave-uniform: nothing to add
    // S^T = K.Q^T: two 16-key halves; D layout: key = t * 16 + g4 * 4 + i, query column l16
    u32x4 ka[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) ka[t][kb] = *(const u32x4*)&sh.k[t * 16 + l16][kb * 32 + g4 * 8];
#pragma unroll
    for (int h = 0; h < HPW; ++h) {
      f32x4 sc[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) d = mfma16x16x32(ka[t][kb], qreg[h][kb], d);
        sc[t] = d;
      }
      float sv[8];
      float mloc = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + t * 16 + g4 * 4 + i;
          const float v = !MASKED || (qok && key <= pq) ? sc[t][i] * scale_log2 : -INFINITY;
          sv[t * 4 + i] = v;
          mloc = fmaxf(mloc, v);
        }
      mloc = max_rows32(max_rows16(mloc));
      const float m_new = fmaxf(m_run[h], mloc);
      const float msafe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = exp2_hw(m_run[h] - msafe);
      float psum = 0.f;
      unsigned pk[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float pa = exp2_hw(sv[2 * jj] - msafe);
        const float pb = exp2_hw(sv[2 * jj + 1] - msafe);
        psum += pa + pb;
        pk[jj] = pk_bf16(pa, pb);
      }
      psum = sum_rows32(sum_rows16(psum));
      l_run[h] = l_run[h] * alpha + psum;
      m_run[h] = m_new;
      const u32x4 pB = {pk[0], pk[1], pk[2], pk[3]};
      // O^T += V^T.P^T; V^T operand: dims dt * 16 + l16, keys g4 * 4 .. + 3 and
      // 16 + g4 * 4 .. + 3 (the keys the lane's P values belong to)
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const u32x2 lo = lds_read_tr16(&sh.v[trow][dt * 16 + tcol]);
        const u32x2 hi = lds_read_tr16(&sh.v[16 + trow][dt * 16 + tcol]);
        acc[h][dt] *= alpha;
        acc[h][dt] = mfma16x16x32(u32x4{lo.x, lo.y, hi.x, hi.y}, pB, acc[h][dt]);
      }
    }
  };
  // blocks whose last key is at or before the workgroup's first query position: no mask; then the
  // blocks that reach into the tile
  const int nfull = min(nblk, (p0 + 1) / KB);
  fetch(0);
  for (int blk = 0; blk < nfull; ++blk) block(blk, std::integral_constant<bool, false>{});
  for (int blk = nfull; blk < nblk; ++blk) block(blk, std::integral_constant<bool, true>{});
  // out: O^T D layout: dim dt * 16 + g4 * 4 + i, token column l16
  if (!qok) return;
#pragma unroll
  for (int h = 0; h < HPW; ++h) {
    bf16* orow = last_only ? out + ((size_t)b * NH + head0 + h) * HD
                           : out + ((size_t)(s0 + pq) * NH + head0 + h) * HD;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) orow[dt * 16 + g4 * 4 + i] = f2bf(acc[h][dt][i] / l_run[h]);
  }
}

// ---------------------------------------------------------------------------------------------
// The same attention for G = 4 with 32 queries per wave and 64-key blocks: wave w takes query head w % 4 of
// tokens 32 (w / 4) .. + 31 of its workgroup's tile, 8 waves (64 tokens, one workgroup per CU) or 4 (32
// tokens, two per CU).
//
// What bounds it: MFMA and the softmax's VALU work are about equal (per wave and block 32 MFMAs of
// 32x32x16, 1,024 cycles, against ~220 VALU instructions), and every K / V operand byte read from LDS
// feeds 32 queries (16 in the kernel above). So the two waves of a SIMD should be in different parts of
// a block: two workgroups of 4 waves are by themselves; the halves of an 8-wave workgroup (waves w and
// w + 4 share a SIMD) run one phase apart: while waves 0 - 3 multiply (P.V of block j and K.Q of block
// j + 1), waves 4 - 7 do the softmax of block j, then the other way round, one barrier a phase. S and P
// of one block are all that a wave holds. K and V have 3 LDS buffers each (2 for 4 waves), filled by
// LDS-DMA four phases (a block) ahead; asm, so that the compiler ties no LDS read to the loads in
// flight; the waits are made by hand. The operand reads of a phase run ahead of its MFMAs (left in the
// compiler's order 671 against 617 us at 8,192 tokens). The kv head is the grid's fast dimension: the
// heaviest tiles of every head go first (with the tiles fast, the last head's heavy tiles started last:
// 617 against 527 us), and each XCD's L2 sees the keys of NKV / 8 heads.
// A query's bits do not depend on the tile or the number of waves.
//
// Graph-timed on MI355X, us, with 16 queries per wave and 32-key blocks (the kernel that this one
// replaced) / this one, in turn on one card: 131 tokens 7.2 / 7.9, 512 16.1 / 15.8, 1,000 32.4 / 26.2, 2,048
// 88 / 55, 16 prompts of 64 - 2,048 459 / 358, 4,096 239 / 146, 8,192 806 / 529 (1.04 PFLOP/s of causal
// attention, MFMA 53% and VALU 57% busy). The shortest prompts lose: three 64-key blocks one after the
// other on 40 workgroups, where 72 had five of 32 keys. 4 waves / 8 waves (another card): 512 16.7 / 21.9,
// 1,000 27.7 / 32.6, 2,048 57.6 / 63.5, 16 prompts 292 / 302, 4,096 174 / 157, 8,192 549 / 525: 8 waves
// from 4,096 tokens per prompt on.
//
// 32x32x16 layouts: S^T lane l holds query l % 32, keys 8 (i / 4) + 4 (l / 32) + i % 4 of 32; those are
// the keys its P values keep in the P.V contraction, so P never leaves the lane and the V^T operand
// reads (transposing) fetch those keys. LDS rows are 256 bytes, 16-byte chunk c of row r at c ^ (r % 16)
// for K (an operand read: one chunk of 32 rows), c ^ 4 (r % 4) for V (4 rows, 4 chunks a half wave):
// no bank conflicts counted.
constexpr int PP_KB = 64;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// LDS bytes: 3 buffers of K and of V for 8 waves, 2 for 4
constexpr int pp_lds(int nw) { return (nw == 8 ? 3 : 2) * 2 * PP_KB * HD * 2; }

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

template <int NW>
__global__ void __launch_bounds__(64 * NW, 2)
flash_prefill_pp_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
                        const int* __restrict__ seq_start, int B, int T, bf16* __restrict__ out, int NH, int NKV,
                        int cap, int last_only, float scale_log2) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char pp_smem[];
  constexpr int TQ = 8 * NW, G = 4, NB = NW == 8 ? 3 : 2, BUF = PP_KB * HD, IPW = 16 / NW;
  bf16* const shk = (bf16*)pp_smem;
  bf16* const shv = shk + NB * BUF;
  int b = 0, p0 = 0;
  const int tile = blockIdx.x / NKV, kvh = blockIdx.x - tile * NKV;   // one dimension: a grid's y ends at 65,535
  if (!tile_of(seq_start, B, tile, last_only != 0, TQ, b, p0)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const bool late = wave >= 4;                                  // one phase behind (waves w, w + 4 share a SIMD)
  const int head = kvh * G + (wave & 3);
  const int s0 = seq_start[b], len = seq_start[b + 1] - s0;
  if (s0 < 0 || len <= 0 || s0 + len > T || len > cap) return;   // inconsistent offsets: no access
  const int pq = p0 + (late ? 32 : 0) + l32;                    // this lane's query position
  const bool qok = last_only ? pq == len - 1 : pq < len;
  const size_t qrow = last_only ? b : s0 + pq;
  const int nblk = (min(p0 + TQ, len) - 1) / PP_KB + 1;
  u32x4 qreg[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks)
    qreg[ks] = qok ? *(const u32x4*)(q + (qrow * NH + head) * HD + ks * 16 + h * 8) : u32x4{0u, 0u, 0u, 0u};
  const size_t kvbase = ((size_t)b * NKV + kvh) * cap * HD;
  const rsrc_t kr = make_rsrc(kc + kvbase, (unsigned)len * HD * 2), vr = make_rsrc(vc + kvbase, (unsigned)len * HD * 2);
  const unsigned lds_k = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) bf16*)shk);
  const unsigned lds_v = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) bf16*)shv);
  // DMA: instruction i fills rows 4 i .. 4 i + 3 of a buffer; wave w issues IPW of them. Rows past the
  // prompt are out of the range and land as zeros (masked, 0 x 0); blocks past the last repeat it (not used).
  auto dma = [&](rsrc_t r, unsigned voff, unsigned lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "s"(lds) : "m0", "memory");
  };
  const int drow = 4 * IPW * wave + (lane >> 4), dc = lane & 15;
  auto issue_k = [&](int j, int buf) {
    const int key0 = min(j, nblk - 1) * PP_KB;
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int r = drow + 4 * i;
      dma(kr, (unsigned)(key0 + r) * HD * 2 + (dc ^ (r & 15)) * 16, lds_k + buf * (BUF * 2) + (IPW * wave + i) * 1024);
    }
  };
  auto issue_v = [&](int j, int buf) {
    const int key0 = min(j, nblk - 1) * PP_KB;
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int r = drow + 4 * i;
      dma(vr, (unsigned)(key0 + r) * HD * 2 + (dc ^ (4 * (r & 3))) * 16, lds_v + buf * (BUF * 2) + (IPW * wave + i) * 1024);
    }
  };
  auto phase_end = [&] {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto landed = [&] {                                           // all but this wave's latest 4 loads
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  };
  // operand addresses (elements) inside a buffer
  int ka[8], va[4];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) ka[ks] = l32 * HD + (((ks * 2 + h) ^ (l32 & 15)) << 3);
  {
    const int l16 = lane & 15, g = (lane >> 4) & 1, r = 4 * h + (l16 >> 2);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int col = d * 32 + g * 16 + 4 * (l16 & 3);
      va[d] = r * HD + (((col >> 3) ^ (4 * (r & 3))) << 3) + (col & 7);
    }
  }
  f32x16 acc[4], sc[2];
  u32x4 pk[4];
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.f;
  auto qk = [&](int buf) {                                      // S^T of a block
    const bf16* kb = shk + buf * BUF;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[t][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) sc[t] = mfma32(*(const u32x4*)&kb[t * 32 * HD + ka[ks]], qreg[ks], sc[t]);
    }
  };
  // O^T += V^T.P^T of a block, and (QK) S^T of the next one. The operand reads run two key steps ahead of
  // their MFMAs: left alone, the compiler reads each operand right before its MFMA and waits for it.
  auto pv = [&](int bv, int bk, auto with_qk, auto nsteps) {
    constexpr bool QK = decltype(with_qk)::value;
    constexpr int NS = decltype(nsteps)::value;                 // 16-key steps
    const bf16* vb = shv + bv * BUF;
    u32x4 vf[NS][4];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const u32x2 lo = lds_read_tr16(&vb[t * 16 * HD + va[d]]);
        const u32x2 hi = lds_read_tr16(&vb[(t * 16 + 8) * HD + va[d]]);
        vf[t][d] = u32x4{lo.x, lo.y, hi.x, hi.y};
      }
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[d] = mfma32(vf[t][d], pk[t], acc[d]);
    if constexpr (QK) qk(bk);
    __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);         // V of steps 0 and 1
#pragma unroll
    for (int i = 0; i < (NS - 2) * 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);        // V of steps 2 and 3
    }
    if constexpr (QK) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);      // K
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
    } else {
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    }
  };
  auto softmax = [&](int j) {
    if (j * PP_KB + PP_KB - 1 > p0 + (late ? 32 : 0)) {         // the block reaches past the wave's first query
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (j * PP_KB + t * 32 + 8 * (i / 4) + 4 * h + i % 4 > pq) sc[t][i] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[t][i]);
    mx = max_rows32(mx);                                        // raw scores
    const bool up = mx > m_run;
    // A row's maximum is -inf until it meets a finite score (key 0 is always seen, but its score may
    // overflow): 0 in its place gives such keys weight 0 and no inf - inf.
    auto finite = [](float m) { return m == -INFINITY ? 0.f : m; };
    if (__any(up)) {
      const float m_old = m_run;
      m_run = up ? mx : m_run;
      const float alpha = exp2_hw((m_old - finite(m_run)) * scale_log2);   // 1 in rows that keep theirs
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] *= alpha;
    }
    const float mscl = finite(m_run) * scale_log2;
    float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float pa = exp2_hw(__builtin_fmaf(sc[t][i], scale_log2, -mscl));
        const float pb = exp2_hw(__builtin_fmaf(sc[t][i + 1], scale_log2, -mscl));
        ps[(i / 2) & 3] += pa + pb;
        pk[t * 2 + i / 8][(i & 7) / 2] = pk_bf16(pa, pb);
      }
    l_run += sum_rows32((ps[0] + ps[1]) + (ps[2] + ps[3]));
  };

  const std::integral_constant<bool, true> next{};
  const std::integral_constant<int, 4> all{};
  // The last block: a wave whose queries lie in its first half leaves the second, whose keys they do not
  // see, out, so that no infinite value there meets their weight 0.
  auto pv_last = [&](int bv) {
    const std::integral_constant<bool, false> final{};
    if ((p0 & 32) || late) pv(bv, 0, final, all);
    else pv(bv, 0, final, std::integral_constant<int, 2>{});
  };
  issue_k(0, 0);
  issue_k(1, 1);
  issue_v(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  phase_end();
  if constexpr (NW == 4) {                                      // two workgroups per CU overlap by themselves
    qk(0);
    for (int j = 0; j + 1 < nblk; ++j) {
      softmax(j);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      phase_end();                                              // block j - 1 is read, V(j) and K(j + 1) landed
      issue_k(j + 2, j & 1);
      issue_v(j + 1, (j + 1) & 1);
      pv(j & 1, (j + 1) & 1, next, all);
    }
    softmax(nblk - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    phase_end();
    pv_last((nblk - 1) & 1);
  } else {
    issue_k(2, 2);
    issue_v(1, 1);
    int b0 = 0, b1 = 1, b2 = 2;                                   // buffers of blocks j, j + 1, j + 2 (K and V)
    auto turn = [&] {
      const int t = b0;
      b0 = b1;
      b1 = b2;
      b2 = t;
    };
    if (!late) {
      qk(0);
      phase_end();
      for (int j = 0; j + 1 < nblk; ++j) {
        softmax(j);
        landed();
        phase_end();
        issue_k(j + 3, b0);
        issue_v(j + 2, b2);
        pv(b0, b1, next, all);
        phase_end();
        turn();
      }
      softmax(nblk - 1);
      landed();
      phase_end();
      pv_last(b0);
      phase_end();
    } else {
      phase_end();
      qk(0);
      landed();
      phase_end();
      for (int j = 0; j + 1 < nblk; ++j) {
        issue_k(j + 3, b0);
        issue_v(j + 2, b2);
        softmax(j);
        phase_end();
        pv(b0, b1, next, all);
        landed();
        phase_end();
        turn();
      }
      softmax(nblk - 1);
      phase_end();
      pv_last(b0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // no load into LDS outlives the wave
  if (!qok) return;
  const float inv = 1.0f / l_run;
  bf16* orow = out + (qrow * NH + head) * HD;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; i += 4)
      *(u32x2*)(orow + d * 32 + 2 * i + 4 * h) = u32x2{pk_bf16(acc[d][i] * inv, acc[d][i + 1] * inv),
                                                      pk_bf16(acc[d][i + 2] * inv, acc[d][i + 3] * inv)};
}

}  // namespace pf
}  // namespace dd

// ------------------------------------------------------------------------------------------
// C ABI
#include "api.h"

using namespace dd;

DD_API int dd_qkv_post_prefill(const void* qkv, const void* qn, const void* kn, const void* cos_t,
                               const void* sin_t, int rope_rows, const int* seq_start, int B, int T,
                               int last_only, void* q_out, void* kc, void* vc, int NH, int NKV,
                               int HD, int cap, float eps, int* err, hipStream_t stream) {
  DD_REQUIRE(qkv && qn && kn && cos_t && sin_t && seq_start && q_out && kc && vc);
  DD_REQUIRE(HD == 128 && B >= 1 && T >= 1 && NKV >= 1 && NH >= NKV && NH % NKV == 0);
  DD_REQUIRE(cap >= 1 && rope_rows >= 1);
  DD_REQUIRE((long long)T * (NH + 2 * NKV) * HD < (1ll << 40));
  const int nheads = NH + 2 * NKV;
  const int hpw = T <= 4096 ? 4 : 8;     // heads per workgroup, see qkv_prefill_kernel
  hipLaunchKernelGGL(pf::qkv_prefill_kernel,
                     dim3((T + pf::QKV_TPW - 1) / pf::QKV_TPW, (nheads + hpw - 1) / hpw), dim3(256), 0,
                     stream, (const bf16*)qkv, (const bf16*)qn, (const bf16*)kn, (const bf16*)cos_t,
                     (const bf16*)sin_t, seq_start, B, T, last_only, (bf16*)q_out, (bf16*)kc,
                     (bf16*)vc, NH, NKV, cap, rope_rows, eps, err, hpw);
  return launch_status();
}

DD_API int dd_attn_prefill(const void* q, const void* kc, const void* vc, const int* seq_start,
                           int B, int T, int last_only, void* out, int NH, int NKV, int HD, int cap,
                           hipStream_t stream) {
  DD_REQUIRE(q && kc && vc && seq_start && out);
  DD_REQUIRE(HD == 128 && B >= 1 && T >= 1 && NKV >= 1 && NH >= NKV && NH % NKV == 0);
  const int G = NH / NKV;
  DD_REQUIRE((G == 1 || G == 2 || G == 4 || G == 8) && cap >= 1);
  DD_REQUIRE(aligned16(q) && aligned16(kc) && aligned16(vc));
  // HD^-0.5 log2(e), formed in double and rounded once (the reference passes the product of two
  // Python floats to a float32 kernel argument)
  const float scale_log2 = (float)(1.0 / sqrt((double)HD) * 1.4426950408889634);
  // 4 waves: HPW heads x (16 NTT tokens) per wave group; tiles per launch at most T / TQ + B
  auto launch = [&](auto kern, int TQ, int nw) {
    const int ntiles = last_only ? B : T / TQ + B;
    hipLaunchKernelGGL(kern, dim3(ntiles, NKV), dim3(64 * nw), 0, stream, (const bf16*)q,
                       (const bf16*)kc, (const bf16*)vc, seq_start, B, T, (bf16*)out, NH, NKV, cap,
                       last_only, scale_log2);
  };
  hipError_t attr = hipSuccess;
  auto launch_pp = [&](int nw) {
    static std::atomic<unsigned long long> done4, done8;
    auto kern = nw == 8 ? pf::flash_prefill_pp_kernel<8> : pf::flash_prefill_pp_kernel<4>;
    attr = allow_lds((const void*)kern, pf::pp_lds(nw), nw == 8 ? done8 : done4);
    if (attr != hipSuccess) return;
    const int ntiles = last_only ? B : T / (8 * nw) + B;
    hipLaunchKernelGGL(kern, dim3((unsigned)ntiles * NKV), dim3(64 * nw), pf::pp_lds(nw), stream, (const bf16*)q, (const bf16*)kc,
                       (const bf16*)vc, seq_start, B, T, (bf16*)out, NH, NKV, cap, last_only, scale_log2);
  };
  switch (G) {
    case 1: launch(pf::flash_prefill_kernel<1, 4, 4, DD_PF_MINB>, 64, 4); break;
    case 2: launch(pf::flash_prefill_kernel<2, 4, 4, DD_PF_MINB>, 64, 4); break;
    case 4:
      launch_pp(!last_only && T / B >= 4096 ? 8 : 4);
      break;
    default: launch(pf::flash_prefill_kernel<2, 1, 4, DD_PF_MINB>, 16, 4); break;   // G = 8
  }
  return attr != hipSuccess ? (int)attr : launch_status();
}
