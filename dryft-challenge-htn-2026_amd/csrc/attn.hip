// Split-KV GQA decode attention with an in-kernel log-sum-exp combine, gfx950.
//
//   out[b*W + s][(kvh*G + g)*HD + d] = softmax_j(q . k_j * HD^-0.5) . v_j
//   over keys j = 0 .. pos[b] + s  of kv head kvh (query row r = s*G + g of that head)
//
// Inputs  q  [B, NKV, W, G, HD] bf16      kc, vc [B, NKV, cap, HD] bf16 (zero-initialised cache)
//         pos int64, row b at pos[b * pos_stride]
// Output  out [B*W, NH*HD] bf16
//
// Two work splits. attn_stream_kernel (below; up to 4 query rows per pair, batches up to 512): equal
// shares of the batch's key blocks. attn_decode_kernel (verify rows, larger batches, an explicit chunk):
// one workgroup per (b*NKV + kvh, split) over a fixed key chunk of C keys, so ragged
// lengths balance across the grid (a split past the row's length exits at once). Inside, the 4
// waves take 32-key blocks round-robin and keep their own online-softmax state:
//   S^T = K . Q^T   on MFMA 16x16x32 (A = 16 keys x 32 dims loaded straight from HBM,
//                   B = Q^T held in registers), fp32 scores in the log2 domain;
//   O^T += V^T . P^T  on MFMA (A = V^T read transposed from an LDS copy of the V block,
//                   B = P^T, which is exactly the lanes' own S^T accumulators rounded to bf16 --
//                   the key order inside the contraction is permuted to make that local).
// P is rounded to bf16 before PV and the running sum l uses the fp32 P (the reference's fused
// kernel does the same, fused.py:511-525). The waves merge through LDS; a single-split row
// writes bf16 directly, otherwise fp32 partials (acc, m, l) go to ws and the last split to
// arrive (per (b, kvh) counter) combines them in split order and resets the counter.
#include <type_traits>

#include "common.h"

namespace dd {

constexpr int ATT_THREADS = 256;
constexpr int ATT_WAVES = 4;
constexpr int HD = 128;
constexpr int VROW = HD + 8;  // padded LDS row (elements) for the V block: 272 bytes

struct AttnShared {
  union {
    bf16 v[ATT_WAVES][32][VROW];                // per-wave V block
    float mrg[ATT_WAVES][16][HD];               // wave partial O (one 16-row block at a time)
  } u;
  float ms[ATT_WAVES][16];
  float ls[ATT_WAVES][16];
  int last;
};

template <int RB>
__global__ void __launch_bounds__(ATT_THREADS)
attn_decode_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kc,
                   const bf16* __restrict__ vc, const int64_t* __restrict__ pos, int pos_stride,
                   bf16* __restrict__ out, float* __restrict__ ws, int* __restrict__ counters,
                   int W, int G, int NKV, int cap, int chunk, int nsplit_max, float scale_log2) {
  __shared__ AttnShared sh;
  const int bk = blockIdx.x;
  const int split = blockIdx.y;
  const int b = bk / NKV, kvh = bk % NKV;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  const int R = W * G;
  const int64_t p0 = pos[(size_t)b * pos_stride];
  const int L = (int)min<int64_t>(p0 + W, (int64_t)cap);  // keys 0 .. L-1 exist
  const int nsplit = (L + chunk - 1) / chunk;
  if (split >= nsplit) return;
  const int start = split * chunk;
  const int end = min(start + chunk, L);

  const bf16* qb = q + (size_t)bk * R * HD;
  const bf16* kb_ = kc + (size_t)bk * cap * HD;
  const bf16* vb_ = vc + (size_t)bk * cap * HD;

  // Q^T operand (B of the S^T MFMA): lane holds q[row rb*16 + l16][kb*32 + g4*8 .. +8]
  u32x4 qreg[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = rb * 16 + l16;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      if (row < R) qreg[rb][kb] = ld16(qb + (size_t)row * HD + kb * 32 + g4 * 8);
      else qreg[rb][kb] = u32x4{0u, 0u, 0u, 0u};
    }
  }
  // causal limit of this lane's query row (as a key index, inclusive)
  int lim[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = rb * 16 + l16;
    lim[rb] = (int)p0 + (row < R ? row : R - 1) / G;
  }

  f32x4 acc[RB][8];
  float m_run[RB], l_run[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    m_run[rb] = -INFINITY;
    l_run[rb] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[rb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  bf16(*vs)[VROW] = sh.u.v[wave];
  const int nblk = (end - start + 31) >> 5;
  for (int bi = wave; bi < nblk; bi += ATT_WAVES) {
    const int j0 = start + bi * 32;
    // K operand loads: 2 tiles of 16 keys x 4 dim blocks
    u32x4 kreg[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      int key = j0 + t * 16 + l16;
      key = key < cap ? key : cap - 1;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) kreg[t][kb] = ld16(kb_ + (size_t)key * HD + kb * 32 + g4 * 8);
    }
    // V block -> registers -> LDS (natural [key][dim] layout)
    u32x4 vreg[8];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int c = it * 64 + lane;
      int key = j0 + (c >> 4);
      key = key < cap ? key : cap - 1;
      vreg[it] = ld16(vb_ + (size_t)key * HD + (c & 15) * 8);
    }
    // S^T tiles
    f32x4 sc[2][RB];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) d = mfma16x16x32(kreg[t][kb], qreg[rb][kb], d);
        sc[t][rb] = d;
      }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int c = it * 64 + lane;
      *(u32x4*)&vs[c >> 4][(c & 15) * 8] = vreg[it];
    }
    // online softmax per 16-row block; P^T operand packed as bf16 pairs
    u32x4 pB[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float sv[8];
      float mloc = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = j0 + t * 16 + g4 * 4 + i;
          const bool ok = key < end && key <= lim[rb];
          const float v = ok ? sc[t][rb][i] * scale_log2 : -INFINITY;
          sv[t * 4 + i] = v;
          mloc = fmaxf(mloc, v);
        }
      mloc = fmaxf(mloc, __shfl_xor(mloc, 16, 64));
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
      const float m_new = fmaxf(m_run[rb], mloc);
      const float msafe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = exp2_hw(m_run[rb] - msafe);
      float psum = 0.f;
      unsigned pk[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float pa = exp2_hw(sv[2 * j] - msafe);
        const float pb = exp2_hw(sv[2 * j + 1] - msafe);
        psum += pa + pb;
        pk[j] = (unsigned)f2bf(pa) | ((unsigned)f2bf(pb) << 16);
      }
      psum += __shfl_xor(psum, 16, 64);
      psum += __shfl_xor(psum, 32, 64);
      l_run[rb] = l_run[rb] * alpha + psum;
      m_run[rb] = m_new;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[rb][dt] *= alpha;
      pB[rb] = u32x4{pk[0], pk[1], pk[2], pk[3]};
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // O^T += V^T . P^T ; V^T operand: dim dt*16 + l16, keys {g4*4 + i} then {16 + g4*4 + i}
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const int d = dt * 16 + l16;
      unsigned a[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int ka = (j < 2) ? (g4 * 4 + 2 * j) : (16 + g4 * 4 + 2 * (j - 2));
        a[j] = (unsigned)vs[ka][d] | ((unsigned)vs[ka + 1][d] << 16);
      }
      const u32x4 va = {a[0], a[1], a[2], a[3]};
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) acc[rb][dt] = mfma16x16x32(va, pB[rb], acc[rb][dt]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // ---- merge the 4 waves, one 16-row block at a time ----
  const size_t wsrow = HD + 2;
  const rsrc_t wsr = make_rsrc(ws, (unsigned)((size_t)gridDim.x * nsplit_max * R * wsrow * 4));
  for (int rb = 0; rb < RB; ++rb) {
    __syncthreads();  // V staging area is reused for the merge
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) sh.u.mrg[wave][l16][dt * 16 + g4 * 4 + i] = acc[rb][dt][i];
    if (g4 == 0) {
      sh.ms[wave][l16] = m_run[rb];
      sh.ls[wave][l16] = l_run[rb];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * HD; e += ATT_THREADS) {
      const int rr = e / HD, d = e % HD;
      const int row = rb * 16 + rr;
      if (row >= R) continue;
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < ATT_WAVES; ++w) M = fmaxf(M, sh.ms[w][rr]);
      const float Ms = M == -INFINITY ? 0.f : M;
      float o = 0.f, l = 0.f;
#pragma unroll
      for (int w = 0; w < ATT_WAVES; ++w) {
        const float f = exp2_hw(sh.ms[w][rr] - Ms);
        o += sh.u.mrg[w][rr][d] * f;
        l += sh.ls[w][rr] * f;
      }
      if (nsplit == 1) {
        const int sq = row / G, gq = row % G;
        out[((size_t)b * W + sq) * (NKV * G * HD) + ((size_t)kvh * G + gq) * HD + d] = f2bf(o / l);
      } else {
        const unsigned p = (unsigned)((((size_t)bk * nsplit_max + split) * R + row) * wsrow) * 4;
        stc_f32(wsr, p + d * 4, o);
        if (d == 0) {
          stc_f32(wsr, p + HD * 4, M);
          stc_f32(wsr, p + (HD + 1) * 4, l);
        }
      }
    }
  }
  if (nsplit == 1) return;

  // ---- last split to arrive combines (split order); partials travel through sc1 ----
  if (!arrive_last(counters + bk, nsplit, &sh.last)) return;
  for (int e = threadIdx.x; e < R * HD; e += ATT_THREADS) {
    const int row = e / HD, d = e % HD;
    const unsigned p = (unsigned)(((size_t)bk * nsplit_max * R + row) * wsrow) * 4;
    const unsigned sstride = (unsigned)(R * wsrow) * 4;
    float M = -INFINITY;
    for (int sp = 0; sp < nsplit; ++sp) M = fmaxf(M, ldc_f32(wsr, p + sp * sstride + HD * 4));
    float o = 0.f, l = 0.f;
    for (int sp = 0; sp < nsplit; ++sp) {
      const unsigned ps = p + sp * sstride;
      const float f = exp2_hw(ldc_f32(wsr, ps + HD * 4) - M);
      o += ldc_f32(wsr, ps + d * 4) * f;
      l += ldc_f32(wsr, ps + (HD + 1) * 4) * f;
    }
    const int sq = row / G, gq = row % G;
    out[((size_t)b * W + sq) * (NKV * G * HD) + ((size_t)kvh * G + gq) * HD + d] = f2bf(o / l);
  }
}

// ---------------------------------------------------------------------------------------------
// Decode rows of up to 4 queries per kv head (W * G <= 4, the decode step of G <= 4) in a batch of up
// to 512: the same arithmetic with the work dealt in equal shares. Where a pair is cut, and with it the last
// bits of its row, depends on the lengths of the whole batch (with fixed chunks it depends on B, NKV and the
// capacity alone); the same batch gives the same bits.
//
// What bounds it: the K/V stream. The fixed key chunks above leave the CUs unevenly loaded on ragged
// batches, every chunk starts with an empty pipeline, and a pair of many chunks is combined by one
// workgroup, one chunk after the other. Here one workgroup of 8 waves per CU takes an equal contiguous
// range of all (pair, 32-key block) units, found from the positions on the device, and each wave an
// equal contiguous part of it. A wave always has the next block in flight, across pairs too: K in a
// second set of operand registers, V by LDS-DMA into the other of two swizzled LDS buffers (read
// transposed), 16 KB per wave, 128 KB per CU. Short batches use as many workgroups as give every wave
// a few blocks. A pair inside a wave's range is written at once; the others merge through LDS and, where
// they lie in several workgroups, through fp32 partials that the last one to arrive adds in workgroup
// order. Graph-timed on MI355X (us, fixed chunks / equal shares; the K/V bytes at 7 TB/s): 16
// sequences of 512 - 8,192 keys 75.5 / 48.6 (35.0), 16 of 576 - 2,560 42.4 / 28.9 (14.6), 64 of 577
// 42.2 / 32.3 (21.6), 32 of 577 28.4 / 20.5 (10.8), one of 8,192 80 / 18.4, one of 513 13.4 / 10.6.
// About 10 us of each are the launch, the positions, the first loads and the combine. MFMA 2.8% and VALU 10%
// busy at the first of these, 5.2 TB/s; 19% of the LDS cycles are bank conflicts, which cost it nothing.
constexpr int STR_WAVES = 8;
// Fewest blocks per workgroup: fewer workgroups mean fewer partials to combine, more waves with a
// block a shorter stream. One sequence of 513 keys: at 4 11.4 us, at 8 13.8, at 16 17.8;
// four of 300 - 2,000 keys 15.8, 17.3, 20.7.
constexpr int STR_MIN = 4;
constexpr int STR_THREADS = 64 * STR_WAVES;
constexpr int STR_R = 4;                          // query rows per pair
constexpr int STR_B = 512;                        // most sequences

struct StreamShared {
  bf16 v[STR_WAVES][2][32 * HD];                  // V blocks; v[w][0] holds the wave's last partial afterwards
  float o[STR_WAVES][STR_R][HD];                  // the wave's first partial (its pair began earlier)
  float ml[STR_WAVES][2][STR_R][2];
  int pair[STR_WAVES][2];                         // pairs of the wave's partials: first, last (-1: none)
  int pre[STR_B + 1];                             // blocks per kv head before sequence b
  int len[STR_B];                                 // keys of sequence b
  int p0[STR_B];                                  // position of its first query (at most the capacity)
  int wsum[STR_WAVES];
  int flag[2];
};

__global__ void __launch_bounds__(STR_THREADS, 1)
attn_stream_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
                   const int64_t* __restrict__ pos, int pos_stride, bf16* __restrict__ out, float* __restrict__ ws,
                   int nslots, int* __restrict__ counters, int B, int W, int G, int NKV, int cap, float scale_log2) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  StreamShared& sh = *(StreamShared*)smem_raw;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int R = W * G;
  // ---- the partition ----
  const int64_t first = tid < B ? pos[(size_t)tid * pos_stride] : -W;
  const int len = (int)max((int64_t)0, min<int64_t>(first + W, (int64_t)cap));
  const int nb = (len + 31) >> 5;
  int inc = nb;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) sh.wsum[wave] = inc;
  if (lane < 2) sh.pair[wave][lane] = -1;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < STR_WAVES; ++w) {
    if (w < wave) before += sh.wsum[w];
    all += sh.wsum[w];
  }
  if (tid < B) {
    sh.pre[tid] = before + inc - nb;
    sh.len[tid] = len;
    sh.p0[tid] = (int)min<int64_t>(first, (int64_t)cap);
  }
  if (tid == 0) sh.pre[B] = all;
  __syncthreads();
  const int total = all * NKV;
  // Partials: slot x for the pair that began before workgroup x, slot nfirst + p for pair p in the
  // workgroup where it begins; o [slots][R][HD], then (m, l) [slots][R].
  const int nfirst = nslots - B * NKV, g = blockIdx.x;
  const int most = nfirst > 0 ? min((int)gridDim.x, nfirst) : (int)gridDim.x;
  const int NG = min(most, (total + STR_MIN - 1) / STR_MIN);
  if (g >= NG) return;
  auto first_of = [&](int gg) { return (int)((long long)total * gg / NG); };
  auto wg_of = [&](int c) { return (int)(((long long)(c + 1) * NG - 1) / total); };
  // block c -> sequence, kv head, block of the pair, blocks of the pair
  auto locate = [&](int c, int& b, int& h, int& j, int& n) {
    int lo = 0, hi = B - 1;
    while (lo < hi) {                             // last sequence with pre * NKV <= c
      const int mid = (lo + hi + 1) >> 1;
      if (sh.pre[mid] * NKV <= c) lo = mid;
      else hi = mid - 1;
    }
    b = __builtin_amdgcn_readfirstlane(lo);
    n = __builtin_amdgcn_readfirstlane(sh.pre[lo + 1] - sh.pre[lo]);
    const int r = c - __builtin_amdgcn_readfirstlane(sh.pre[lo]) * NKV;
    h = r / n;
    j = r - h * n;
  };
  int c0 = first_of(g), c1 = first_of(g + 1);
  if (nfirst == 0) {                              // no room for partials: ranges of whole pairs
    int b, h, j, n;
    locate(c0, b, h, j, n);
    c0 -= j;
    if (c1 < total) {
      locate(c1, b, h, j, n);
      c1 -= j;
    }
    if (c0 == c1) return;
  }
  const int w0 = c0 + (int)((long long)(c1 - c0) * wave / STR_WAVES);
  const int w1 = c0 + (int)((long long)(c1 - c0) * (wave + 1) / STR_WAVES);
  // ---- one block in flight per wave: K operands, V by LDS-DMA ----
  const unsigned lds_v = __builtin_amdgcn_readfirstlane(
      (unsigned)(size_t)(__attribute__((address_space(3))) bf16*)&sh.v[wave][0][0]);
  const int vr = lane >> 4;                       // key within a V instruction's 4
  int b, h, j, n, L, P0;                          // block being requested, its sequence's keys and position
  u32x4 ka[2][4], kb[2][4], qv[4], qn[4];
  auto load_q = [&](u32x4(&dst)[4]) {
    const bf16* qb = q + (size_t)(b * NKV + h) * R * HD;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      dst[k] = l16 < R ? ld16(qb + (size_t)l16 * HD + k * 32 + g4 * 8) : u32x4{0u, 0u, 0u, 0u};
  };
  auto request = [&](u32x4(&kr)[2][4], int buf) {
    const size_t base = (size_t)(b * NKV + h) * cap * HD;
    const rsrc_t krs = make_rsrc(kc + base, (unsigned)L * HD * 2), vrs = make_rsrc(vc + base, (unsigned)L * HD * 2);
    const unsigned k0 = (unsigned)(j * 32 + l16) * HD * 2 + g4 * 16;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int k = 0; k < 4; ++k)                 // keys past the last read 0 (masked)
        kr[t][k] = __builtin_amdgcn_raw_buffer_load_b128(krs, k0 + t * 16 * HD * 2 + k * 64, 0, 2);
#pragma unroll
    for (int i = 0; i < 8; ++i) {                 // 4 keys each; keys past the last: zeros (out of the range)
      const unsigned key = j * 32 + i * 4 + vr;
      const unsigned off = key * HD * 2 + ((l16 ^ (2 * ((i * 4 + vr) & 7))) * 16);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          vrs, (__attribute__((address_space(3))) void*)(size_t)(lds_v + buf * (32 * HD * 2) + i * 1024), 16, off, 0, 0, 2);
    }
  };
  // V^T operand addresses (see lds_read_tr16): dims d * 16 + l16 of keys g4 * 4 .. (and 16 on)
  unsigned vaddr[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int r = g4 * 4 + (l16 >> 2), col = d * 16 + 4 * (l16 & 3);
    vaddr[d] = lds_v + (r * HD + (((col >> 3) ^ (2 * (r & 7))) << 3) + (col & 7)) * 2;
  }
  f32x4 acc[8];
  float m_run, l_run;
  auto clear = [&] {
    m_run = -INFINITY;
    l_run = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  bool begun = false;                             // the segment holds its pair's first block
  auto out_row = [&](int bb, int hh, int row) {
    return out + ((size_t)bb * W + row / G) * ((size_t)NKV * G * HD) + ((size_t)hh * G + row % G) * HD;
  };
  // one block: its operands in kr and buffer buf; the next block (if one follows) goes to kn and the
  // other buffer
  auto step = [&](u32x4(&kr)[2][4], u32x4(&kn)[2][4], auto buf_c, auto follows) {
    constexpr int buf = decltype(buf_c)::value;
    const int cb = b, ch = h, cj = j, cn = n, cL = L, cP = P0;
    constexpr bool MORE = decltype(follows)::value;
    if (cj == 0) begun = true;
    if constexpr (MORE) {
      if (++j == n) {
        j = 0;
        if (++h == NKV) {
          h = 0;
          do { ++b; n = __builtin_amdgcn_readfirstlane(sh.pre[b + 1] - sh.pre[b]); } while (n == 0);
          L = __builtin_amdgcn_readfirstlane(sh.len[b]);
          P0 = __builtin_amdgcn_readfirstlane(sh.p0[b]);
        }
        load_q(qn);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the other buffer's reads are done
      request(kn, buf ^ 1);
      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");    // all but the next block's loads
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    f32x4 sc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k) sc[t] = mfma16x16x32(kr[t][k], qv[k], sc[t]);
    }
    const int lim = min(cP + (l16 < R ? l16 : R - 1) / G, cL - 1) - cj * 32;   // last key of the lane's row
    float sv[8], mloc = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sv[t * 4 + i] = t * 16 + g4 * 4 + i <= lim ? sc[t][i] * scale_log2 : -INFINITY;
        mloc = fmaxf(mloc, sv[t * 4 + i]);
      }
    mloc = max_rows32(max_rows16(mloc));
    const float m_new = fmaxf(m_run, mloc), msafe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_hw(m_run - msafe);
    float psum = 0.f;
    unsigned pk[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float pa = exp2_hw(sv[2 * i] - msafe), pb = exp2_hw(sv[2 * i + 1] - msafe);
      psum += pa + pb;
      pk[i] = pk_bf16(pa, pb);
    }
    psum = sum_rows32(sum_rows16(psum));
    l_run = l_run * alpha + psum;
    m_run = m_new;
    const u32x4 pB = {pk[0], pk[1], pk[2], pk[3]};
#pragma unroll
    for (int d = 0; d < 8; d += 4) {
      u32x2 t[4][2];
      // Written as asm, with its wait: the compiler would wait for every LDS-DMA load in flight (the
      // next block's too) before these reads.
      asm volatile(
          "ds_read_b64_tr_b16 %0, %8 offset:%12\n\tds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
          "ds_read_b64_tr_b16 %2, %9 offset:%12\n\tds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
          "ds_read_b64_tr_b16 %4, %10 offset:%12\n\tds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
          "ds_read_b64_tr_b16 %6, %11 offset:%12\n\tds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(t[0][0]), "=&v"(t[0][1]), "=&v"(t[1][0]), "=&v"(t[1][1]), "=&v"(t[2][0]), "=&v"(t[2][1]),
            "=&v"(t[3][0]), "=&v"(t[3][1])
          : "v"(vaddr[d]), "v"(vaddr[d + 1]), "v"(vaddr[d + 2]), "v"(vaddr[d + 3]), "n"(buf * 32 * HD * 2),
            "n"(buf * 32 * HD * 2 + 16 * HD * 2)
          : "memory");
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[d + i] *= alpha;
        acc[d + i] = mfma16x16x32(u32x4{t[i][0].x, t[i][0].y, t[i][1].x, t[i][1].y}, pB, acc[d + i]);
      }
    }
    if (MORE && cj + 1 < cn) return;              // the segment goes on
    if (begun && cj + 1 == cn) {                  // the whole pair: write it
      if (l16 < R) {
        bf16* o = out_row(cb, ch, l16);
#pragma unroll
        for (int d = 0; d < 8; ++d)
          *(u32x2*)(o + d * 16 + g4 * 4) = u32x2{pk_bf16(acc[d][0] / l_run, acc[d][1] / l_run),
                                                 pk_bf16(acc[d][2] / l_run, acc[d][3] / l_run)};
      }
    } else {                                      // a part of it: leave it in LDS
      const int w = begun ? 1 : 0;
      if (w == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // v[wave][0] is read
      float* o = w == 0 ? &sh.o[wave][0][0] : (float*)sh.v[wave][0];
      if (l16 < R) {
#pragma unroll
        for (int d = 0; d < 8; ++d) *(f32x4*)(o + l16 * HD + d * 16 + g4 * 4) = acc[d];
        if (g4 == 0) {
          sh.ml[wave][w][l16][0] = m_run;
          sh.ml[wave][w][l16][1] = l_run;
        }
      }
      if (lane == 0) sh.pair[wave][w] = cb * NKV + ch;
    }
    clear();
    begun = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) qv[k] = qn[k];
  };
  if (w0 < w1) {
    locate(w0, b, h, j, n);
    L = __builtin_amdgcn_readfirstlane(sh.len[b]);
    P0 = __builtin_amdgcn_readfirstlane(sh.p0[b]);
    load_q(qv);
    request(ka, 0);
    const std::integral_constant<bool, true> more{};
    const std::integral_constant<bool, false> end{};
    const std::integral_constant<int, 0> b0{};
    const std::integral_constant<int, 1> b1{};
    int c = w0;
    for (; c + 2 < w1; c += 2) {
      step(ka, kb, b0, more);
      step(kb, ka, b1, more);
    }
    if (c + 1 < w1) {
      step(ka, kb, b0, more);
      step(kb, ka, b1, end);
    } else {
      step(ka, kb, b0, end);
    }
  }
  __syncthreads();

  // ---- merge the waves' parts of a pair, in wave order ----
  const rsrc_t wsr = make_rsrc(ws, (unsigned)nslots * R * (HD + 2) * 4);
  const unsigned ml0 = (unsigned)nslots * R * HD * 4;
  int sb, shd, sj, sn, eb, eh, ej, en;
  locate(c0, sb, shd, sj, sn);
  locate(c1 - 1, eb, eh, ej, en);
  const int pfirst = sj > 0 ? sb * NKV + shd : -1;            // its pair began in another workgroup
  const bool open = ej + 1 < en;                              // the last pair ends in another one
  const int plast = open && eb * NKV + eh != pfirst ? eb * NKV + eh : -1;
  auto merge = [&](int p) {
    const bool here = p != pfirst && p != plast;              // complete in this workgroup
    const unsigned slot_r = (unsigned)(p == pfirst ? g : nfirst + p) * R;
    for (int e = lane; e < R * (HD / 4); e += 64) {
      const int row = e / (HD / 4), d = (e % (HD / 4)) * 4;
      float M = -INFINITY, l = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < STR_WAVES; ++w)
#pragma unroll
        for (int s = 1; s >= 0; --s)
          if (sh.pair[w][s] == p) M = fmaxf(M, sh.ml[w][s][row][0]);
      const float Ms = M == -INFINITY ? 0.f : M;
#pragma unroll
      for (int w = 0; w < STR_WAVES; ++w)
#pragma unroll
        for (int s = 1; s >= 0; --s)
          if (sh.pair[w][s] == p) {
            const float f = exp2_hw(sh.ml[w][s][row][0] - Ms);
            const float* src = s == 0 ? sh.o[w][row] : (const float*)sh.v[w][0] + row * HD;
            o += *(const f32x4*)(src + d) * f;
            l += sh.ml[w][s][row][1] * f;
          }
      if (here) {
        *(u32x2*)(out_row(p / NKV, p % NKV, row) + d) = u32x2{pk_bf16(o[0] / l, o[1] / l), pk_bf16(o[2] / l, o[3] / l)};
      } else {
        stc_b128(wsr, ((slot_r + row) * HD + d) * 4, __builtin_bit_cast(u32x4, o));
        if (d == 0) {
          stc_f32(wsr, ml0 + (slot_r + row) * 8, M);
          stc_f32(wsr, ml0 + (slot_r + row) * 8 + 4, l);
        }
      }
    }
  };
  if (wave == 0 && pfirst >= 0) merge(pfirst);
  if (sh.pair[wave][1] >= 0) merge(__builtin_amdgcn_readfirstlane(sh.pair[wave][1]));
  if (pfirst < 0 && plast < 0) return;

  // ---- pairs in several workgroups: the last one to arrive adds the partials in workgroup order ----
  auto span = [&](int p, int& ga, int& gb) {
    const int bb = p / NKV, hh = p % NKV, nn = sh.pre[bb + 1] - sh.pre[bb], pc = sh.pre[bb] * NKV + hh * nn;
    ga = wg_of(pc);
    gb = wg_of(pc + nn - 1);
  };
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (lane == 0 && wave < 2) {
    const int p = wave == 0 ? pfirst : plast;
    int last = 0;
    if (p >= 0) {
      int ga, gb;
      span(p, ga, gb);
      last = __hip_atomic_fetch_add(counters + p, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gb - ga;
      if (last) __hip_atomic_store(counters + p, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    sh.flag[wave] = last;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int p = s == 0 ? pfirst : plast;
    if (p < 0 || !sh.flag[s]) continue;
    int ga, gb;
    span(p, ga, gb);
    const int row = tid / HD, d = tid % HD;                   // one element per thread
    if (row >= R) continue;
    float M = -INFINITY, l = 0.f, o = 0.f;
    constexpr int NB = 16;                                    // partials in flight
    for (int x0 = ga; x0 <= gb; x0 += NB) {
      float pm[NB], pl[NB], po[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int x = x0 + i;
        const unsigned sr = (unsigned)(x == ga ? nfirst + p : x) * R + row;   // past the last: not used
        po[i] = x <= gb ? ldc_f32(wsr, (sr * HD + d) * 4) : 0.f;
        pm[i] = x <= gb ? ldc_f32(wsr, ml0 + sr * 8) : 0.f;
        pl[i] = x <= gb ? ldc_f32(wsr, ml0 + sr * 8 + 4) : 0.f;
      }
      float Mb = M;
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (x0 + i <= gb) Mb = fmaxf(Mb, pm[i]);
      const float Ms = Mb == -INFINITY ? 0.f : Mb, f0 = exp2_hw(M - Ms);
      o *= f0;
      l *= f0;
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (x0 + i <= gb) {
          const float f = exp2_hw(pm[i] - Ms);
          o += po[i] * f;
          l += pl[i] * f;
        }
      M = Mb;
    }
    out_row(p / NKV, p % NKV, row)[d] = f2bf(o / l);
  }
}

template __global__ void attn_decode_kernel<1>(const bf16*, const bf16*, const bf16*, const int64_t*, int,
                                               bf16*, float*, int*, int, int, int, int, int, int, float);
template __global__ void attn_decode_kernel<2>(const bf16*, const bf16*, const bf16*, const int64_t*, int,
                                               bf16*, float*, int*, int, int, int, int, int, int, float);

}  // namespace dd

// ------------------------------------------------------------------------------------------
// C ABI
#include "api.h"

using namespace dd;

// Keys per split: aim for ~1024 workgroups over a full cache (256 CUs x 4), in multiples of
// 128 keys (one 32-key block per wave), never below 128.
DD_API int dd_attn_chunk(int B, int NKV, int cap) {
  if (B < 1 || NKV < 1 || cap < 1) return 128;
  const long long keys = (long long)B * NKV * cap;
  long long c = (keys + 1023) / 1024;
  c = (c + 127) / 128 * 128;
  return (int)(c < 128 ? 128 : c);
}

DD_API size_t dd_attn_ws_bytes(int B, int W, int NH, int NKV, int HD, int cap, int chunk) {
  if (chunk <= 0) chunk = dd_attn_chunk(B, NKV, cap);
  if (B < 1 || NKV < 1 || NH < NKV || W < 1 || HD < 1 || cap < 1) return 0;
  const size_t nsplit = (size_t)(cap + chunk - 1) / chunk;
  const size_t R = (size_t)W * (NH / NKV);
  return (size_t)B * NKV * nsplit * R * (HD + 2) * sizeof(float);
}

DD_API int dd_attn_decode(const void* q, const void* kc, const void* vc, const int64_t* pos,
                          int pos_stride, void* out, void* ws, int* counters, int B, int W, int NH,
                          int NKV, int HD, int cap, int chunk, hipStream_t stream) {
  DD_REQUIRE(q && kc && vc && pos && out && ws && counters);
  DD_REQUIRE(HD == 128 && B >= 1 && W >= 1 && NKV >= 1 && NH >= NKV && NH % NKV == 0 && cap >= 1);
  DD_REQUIRE(pos_stride == 0 || pos_stride == 1);
  const int G = NH / NKV;
  DD_REQUIRE(W * G <= 32);
  DD_REQUIRE(aligned16(q) && aligned16(kc) && aligned16(vc));
  if (chunk <= 0) chunk = dd_attn_chunk(B, NKV, cap);
  DD_REQUIRE(chunk % 32 == 0);
  const int nsplit_max = (cap + chunk - 1) / chunk;
  const float scale_log2 = (1.0f / sqrtf((float)HD)) * 1.4426950408889634f;
  dim3 grid(B * NKV, nsplit_max);
  // Up to 4 query rows per pair: equal shares of the whole batch (an explicit other chunk keeps the
  // chunks). The partials lie in the chunks' workspace; where that has one chunk per pair (about 1,000
  // pairs on) the shares are rounded to whole pairs.
  const int cus = cu_count();
  static std::atomic<unsigned long long> done;
  if (W * G <= STR_R && B <= STR_B && chunk == dd_attn_chunk(B, NKV, cap) && cus > 0 &&
      (long long)B * NKV * cap < (1ll << 31) && (long long)cap * HD * 2 < (1ll << 31) &&
      (long long)B * NKV * nsplit_max * W * G * (HD + 2) * 4 < (1ll << 31) &&
      allow_lds((const void*)attn_stream_kernel, (int)sizeof(StreamShared), done) == hipSuccess)
    hipLaunchKernelGGL(attn_stream_kernel, dim3(cus), dim3(STR_THREADS), sizeof(StreamShared), stream,
                       (const bf16*)q, (const bf16*)kc, (const bf16*)vc, pos, pos_stride, (bf16*)out, (float*)ws,
                       B * NKV * nsplit_max, counters, B, W, G, NKV, cap, scale_log2);
  else if (W * G <= 16)
    hipLaunchKernelGGL(attn_decode_kernel<1>, grid, dim3(ATT_THREADS), 0, stream, (const bf16*)q,
                       (const bf16*)kc, (const bf16*)vc, pos, pos_stride, (bf16*)out, (float*)ws,
                       counters, W, G, NKV, cap, chunk, nsplit_max, scale_log2);
  else
    hipLaunchKernelGGL(attn_decode_kernel<2>, grid, dim3(ATT_THREADS), 0, stream, (const bf16*)q,
                       (const bf16*)kc, (const bf16*)vc, pos, pos_stride, (bf16*)out, (float*)ws,
                       counters, W, G, NKV, cap, chunk, nsplit_max, scale_log2);
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// No-allocation variant: the split partials and the per-(row, kv head) counters live in a
// file-scope device array instead of caller workspaces. Each device holds its own copy of the
// array (for the life of the process); host code reaches it only through the address
// hipGetSymbolAddress returns for the current device, looked up once per device.
namespace dd {
constexpr size_t NOALLOC_WS_BYTES = size_t(24) << 20;   // split partials (dd_attn_ws_bytes)
constexpr int NOALLOC_COUNTERS = 4096;                  // B * NKV combine counters
static __device__ __align__(256) unsigned char scratch[NOALLOC_WS_BYTES + NOALLOC_COUNTERS * 4];

__global__ void zero_ints_kernel(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace dd

#include <mutex>

namespace {
constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[NOALLOC_MAX_DEVICES];   // device address of `scratch`, per device

// Address of this device's scratch array. The first call on a device looks it up and clears the
// counters synchronously (so no later call, on any stream, can overlap the clear); a first call
// made while `stream` is being captured into a graph returns hipErrorStreamCaptureUnsupported
// instead, since the clear could only be recorded, not done.
int noalloc_scratch(hipStream_t stream, unsigned char** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES)
    return (int)hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (g_noalloc_ptr[dev] == nullptr) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) return (int)hipErrorInvalidValue;
    if (cap != hipStreamCaptureStatusNone) return (int)hipErrorStreamCaptureUnsupported;
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(dd::scratch));
    if (e != hipSuccess) return (int)e;
    if (ptr == nullptr) return (int)hipErrorInvalidSymbol;
    int* counters = (int*)((unsigned char*)ptr + dd::NOALLOC_WS_BYTES);
    hipLaunchKernelGGL(dd::zero_ints_kernel, dim3((dd::NOALLOC_COUNTERS + 255) / 256), dim3(256),
                       0, stream, counters, dd::NOALLOC_COUNTERS);
    const int st = dd::launch_status();
    if (st != 0) return st;
    e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return (int)e;
    g_noalloc_ptr[dev] = ptr;
  }
  *out = (unsigned char*)g_noalloc_ptr[dev];
  return 0;
}
}  // namespace

DD_API int dd_attn_decode_noalloc(const void* q, const void* kc, const void* vc,
                                  const int64_t* pos, int pos_stride, void* out, int B, int W,
                                  int NH, int NKV, int HD, int cap, hipStream_t stream) {
  DD_REQUIRE(q && kc && vc && pos && out);
  DD_REQUIRE(HD == 128 && B >= 1 && W >= 1 && NKV >= 1 && NH >= NKV && NH % NKV == 0 && cap >= 1);
  DD_REQUIRE(pos_stride == 0 || pos_stride == 1);
  DD_REQUIRE(W * (NH / NKV) <= 32);
  DD_REQUIRE(aligned16(q) && aligned16(kc) && aligned16(vc));
  const int chunk = dd_attn_chunk(B, NKV, cap);
  // the static array bounds the shapes this entry point takes
  if (dd_attn_ws_bytes(B, W, NH, NKV, HD, cap, chunk) > dd::NOALLOC_WS_BYTES ||
      (long long)B * NKV > dd::NOALLOC_COUNTERS)
    return (int)hipErrorOutOfMemory;
  unsigned char* base = nullptr;
  const int e = noalloc_scratch(stream, &base);
  if (e != 0) return e;
  return dd_attn_decode(q, kc, vc, pos, pos_stride, out, base, (int*)(base + dd::NOALLOC_WS_BYTES),
                        B, W, NH, NKV, HD, cap, chunk, stream);
}

