// Skinny linear layers (1 <= M <= 64 activation rows; with the SiLU epilogue up to 96, with the sums up to
// 128) that stream the weights through LDS, gfx950.
//
//   y[m][n] = sum_k x[m][k] * W[n][k]          (F.linear semantics, W row-major [N, K])
//
// with three epilogues: the plain product, SiLU(gate) * up, and fp32 sums for the residual add + norm.
//
// What bounds it: the weight stream. A CU's share of the HBM rate is ~27 bytes / ns and a load takes
// 2 - 3 us under load, so 55 - 80 KB per CU have to be in flight at all times. One workgroup of 8 waves
// per CU keeps them in a ring of LDS stages that LDS-DMA loads (buffer_load_dwordx4 ... lds) fill: a stage
// is 64, 128 or 256 columns (whole 128-byte lines of every row) of the tile's weight rows and of x.
// The stage NST - 1 ahead is requested when a stage is consumed, one barrier a stage; the ring runs on
// over the end of a tile into the next one. W is streamed past the caches (nt), x is kept in them.
//
// Split: every workgroup gets the same number of output rows, so no CU idles in a last round of tiles,
// and computes them whole. Each workgroup then reads all of x; where that outweighs its weights (M > 4
// rows per workgroup) and a second launch follows anyway (residual add + norm: O and down above 40
// rows), S = 2, 4, .. workgroups share S times the rows and each takes a part of K; that launch adds
// their fp32 sums in order. Graph-timed on MI355X (cold weights,
// the launches included, us; before: the register-streaming GEMV up to 16 rows, hipBLASLt and separate
// SiLU / add + norm kernels above):
//   rows               1             4            16            32            48            64
//   QKV           11.2 / 10.3   12.0 / 10.4   14.7 / 10.7   11.4 / 10.9   15.4 / 12.1   15.3 / 13.0
//   O + norm      12.6 / 11.5   15.3 / 11.7   24.2 / 12.5   15.7 / 13.1   15.8 / 14.6   17.8 / 14.9
//   gate/up       30.4 / 22.8   31.8 / 22.3   37.5 / 22.3   29.1 / 23.3   32.6 / 25.8   30.4 / 28.3
//   down + norm   18.8 / 16.9   22.4 / 17.4   33.8 / 18.7   23.4 / 21.1   23.7 / 21.8   31.4 / 23.3
//   lm_head        181 / 122     196 / 122     232 / 128     172 / 144     159 / 160     181 / 175
// About 5 us of each are the launch and the first loads' latency; the lm_head streams at 6.4 TB/s. Equal
// shares of K x tiles for every workgroup (stream-K over 64-row tiles) cost the partials' round trips:
// 13.5 us for QKV at M = 1, 14.8 at 32. The norm by the last workgroup of the same launch took 3 us more
// than its own launch (two hand-offs).
// Above 64 rows x's share of the loads grows (every workgroup reads all of it) and hipBLASLt's larger
// tiles win where nothing else is saved (QKV 15.0 / 15.5 at 80 rows, 18.5 / 20.4 at 131). With the
// epilogues a launch and a pass over the product go too (hipBLASLt and the separate kernel / this one):
//   rows              65            80            96           112           128           144
//   gate/up      37.3 / 35.0   37.3 / 36.1   36.1 / 34.5   35.9 / 37.5   34.2 / 38.4   44.3 / 41.1
//   O + norm     18.8 / 16.5   19.1 / 16.9   19.6 / 18.5   19.1 / 18.9   19.5 / 19.5   18.0 / 20.9
//   down + norm  31.0 / 26.2   32.1 / 27.5   34.4 / 26.9   35.6 / 28.3   36.0 / 28.7   32.6 / 31.4
// so the sums are taken up to 128 rows and SiLU up to 96 (from 129 to 160 rows it is 2 - 7% ahead again,
// hipBLASLt's time being a staircase of its tile heights: not worth a second range). A different first
// stage for each workgroup, so that they do not read the same lines of x at once, gained nothing up to 64
// rows and cost 0.5 us in O and down above.
//
// MFMA 16x16x32: A = 16 weight rows, B = 16 activation rows (x^T), both read from LDS. The 8 waves
// split a stage into (k-steps of 32) x (weight tiles), and every wave multiplies its weight fragments
// with all activation tiles. 16-byte chunks are XOR-swizzled inside an LDS row so that the 16 rows of
// a fragment read meet distinct banks; the DMA picks per lane the source chunk whose swizzled position
// is its own.
#include "common.h"

namespace dd {
namespace lin {

constexpr int THREADS = 512;
constexpr int LDS_MAX = 160 * 1024;

enum { OUT = 0, SILU = 1, PART = 2 };

struct Args {
  const bf16* x;
  const bf16* W;
  bf16* y;                                    // OUT, SILU
  float* ws;                                  // PART: fp32 sums [S][M][N]
  int M, N, K;                                // N: rows of W (SILU: 2 I)
  int nout;                                   // output columns (N; SILU: I)
  int nv;                                     // outputs per tile (rows of W; SILU: features)
  int KT, S, C;                               // stages and chunks (parts of K) per tile, chunks in all
};

// Geometry of one instantiation: BMT activation tiles, NT weight tiles.
template <int BMT, int NT>
struct Geo {
  static constexpr int KS = NT == 1 ? 256 : NT == 2 ? 128 : 64;   // columns per stage
  static constexpr int KW = KS / 32;                       // waves along a stage's k-steps
  static constexpr int NG = 8 / KW;                        // waves along the weight tiles
  static constexpr int NTW = (NT + NG - 1) / NG;           // weight tiles per wave
  static constexpr int CPR = KS / 8;                       // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;                     // rows per DMA instruction
  static constexpr int STAGE_W = NT * 16 * KS * 2;
  static constexpr int STAGE = STAGE_W + BMT * 16 * KS * 2;
  static constexpr int NWI = STAGE_W / 1024, NI = STAGE / 1024;   // DMA instructions: W's, all
  static constexpr int IPW = (NI + 7) / 8;                 // most of them in one wave (others: one less)
  // the k-slices meet in the LDS of the stage just consumed, in PASSES parts
  static constexpr int RTILES = STAGE / 1024 / ((KW - 1) * NG * NTW);
  static constexpr int PASSES = (BMT + RTILES - 1) / RTILES;
  static_assert(RTILES >= 1, "k-slice partials fit a stage");
  static constexpr int NST0 = LDS_MAX / STAGE;
  static constexpr int NST = NST0 > 14 ? 14 : NST0;
  static constexpr int LDS = NST * STAGE;
  // chunk swizzle of LDS row r: 8, 16 or 32 chunks a row
  static __device__ __forceinline__ int swz(int r) { return CPR == 8 ? (r >> 1) & 7 : r & 15; }
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// wait until the loads of `rem` <= R later stages, C a stage, are all that is left
template <int R, int C>
__device__ __forceinline__ void wait_stages(int rem) {
  if constexpr (R == 0) {
    wait_vm<0>();
  } else {
    static_assert(R * C < 63, "vmcnt range");
    if (__builtin_expect(rem >= R, 1)) wait_vm<R * C>();
    else wait_stages<R - 1, C>(rem);
  }
}
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// 64 lanes x 16 bytes from r[voff + soff] to LDS byte address `lds` + 16 lane; the ring's waits are
// made by hand (the address is an integer, so the compiler ties no LDS read to it). AUX 2: streamed
// past the caches.
template <int AUX>
__device__ __forceinline__ void dma16(rsrc_t r, unsigned voff, unsigned soff, unsigned lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(size_t)lds, 16, voff, soff, 0, AUX);
}

// first chunk of workgroup g (C >= G chunks)
__device__ __forceinline__ int chunk0(int C, int G, int g) { return (int)((long long)C * g / G); }
// first unit (tile * KT + stage) of chunk c
__device__ __forceinline__ int unit_of(const Args& a, int c) {
  const int t = c / a.S;
  return t * a.KT + (c - t * a.S) * a.KT / a.S;
}

template <int BMT, int NT, int MODE>
__global__ void __launch_bounds__(THREADS, 1) linear_kernel(const Args a) {
  using Z = Geo<BMT, NT>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int G = gridDim.x, g = blockIdx.x;
  int chunk = chunk0(a.C, G, g);
  const int u0 = unit_of(a, chunk), u1 = unit_of(a, chunk0(a.C, G, g + 1));
  const int kslice = wave % Z::KW, ng = wave / Z::KW;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(
      (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem);

  // ---- DMA side: instruction i of a stage (wave i % 8) fills LDS rows i RPI .. of W, then of x ----
  // Rows past M, and weight rows past the tile's last, lie outside the buffers' ranges: those lanes
  // fetch nothing and land zeros, and the outputs of such rows are not stored. So every wave issues the
  // same number of loads in every stage, which is what the waits count.
  const rsrc_t xr = make_rsrc(a.x, (unsigned)a.M * a.K * 2);
  const int ni = (Z::NI - wave + 7) / 8;                               // this wave's instructions
  unsigned off[Z::IPW];
#pragma unroll
  for (int j = 0; j < Z::IPW; ++j) {
    const int i = wave + 8 * j;
    const int r = (i < Z::NWI ? i : i - Z::NWI) * Z::RPI + lane / Z::CPR;
    // SILU: a 16-row weight tile is 8 gate rows, then their 8 up rows
    const int row = MODE == SILU && i < Z::NWI ? (r >> 4) * 8 + (r & 7) + ((r >> 3) & 1) * a.nout : r;
    off[j] = (unsigned)row * a.K * 2 + (lane % Z::CPR ^ Z::swz(r)) * 16;
  }
  rsrc_t wr = make_rsrc(a.W, 0);
  int it = u0 / a.KT, ik = u0 - it * a.KT, islot = 0, ui = u0;
  auto aim = [&] {                                                     // at tile `it`
    const int n0 = it * a.nv, left = min(a.nv, a.nout - n0);
    const int rows = MODE == SILU ? a.nout + left : left;
    wr = make_rsrc((const unsigned char*)a.W + (size_t)n0 * a.K * 2, (unsigned)rows * a.K * 2);
  };
  auto issue = [&] {
    const unsigned so = (unsigned)(ik * Z::KS * 2), ld = lds0 + islot * Z::STAGE;
#pragma unroll
    for (int j = 0; j < Z::IPW; ++j) {
      const int i = wave + 8 * j;
      if (i < Z::NWI) dma16<2>(wr, off[j], so, ld + i * 1024);
      else if (i < Z::NI) dma16<0>(xr, off[j], so, ld + i * 1024);
    }
    islot = islot + 1 == Z::NST ? 0 : islot + 1;
    ++ui;
    if (++ik == a.KT) {
      ik = 0;
      ++it;
      if (ui < u1) aim();
    }
  };

  // ---- MFMA side: wave (kslice, ng) takes k-step kslice of weight tiles ng, ng + NG ----
  auto nt_of = [&](int n) { return ng + n * Z::NG; };
  auto frag = [&](int r) { return r * Z::KS * 2 + (((kslice * 4 + g4) ^ Z::swz(r)) * 16); };
  f32x4 acc[Z::NTW][BMT];
  auto clear = [&] {
#pragma unroll
    for (int n = 0; n < Z::NTW; ++n)
#pragma unroll
      for (int m = 0; m < BMT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  // epilogue of part s of tile t; the k-slice-0 waves hold its sums: output nt * 16 + g4 * 4 + i of row m * 16 + l16
  auto finish = [&](int t, int s) {
    if (kslice != 0) return;
    const int n0 = t * a.nv, left = min(a.nv, a.nout - n0);
    const bool al = a.nout % 4 == 0 && a.nv % 4 == 0;                  // 8-byte accesses of 4 outputs
#pragma unroll
    for (int n = 0; n < Z::NTW; ++n)
#pragma unroll
      for (int m = 0; m < BMT; ++m) {
        f32x4 v = acc[n][m];
        const int row = m * 16 + l16;
        int c = nt_of(n) * 16 + g4 * 4;
        if (MODE == SILU) {                                            // up values lie 32 lanes on
          c = nt_of(n) * 8 + (g4 & 1) * 4;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float up = __shfl_xor(v[i], 32, 64), gg = rbf(v[i]);
            v[i] = rbf(gg / (1.0f + expf(-gg))) * rbf(up);
          }
          if (g4 >= 2) continue;
        }
        if (row >= a.M || c >= left) continue;
        const size_t at = (size_t)row * a.nout + n0 + c;
        if (MODE == PART) {
          float* dst = a.ws + (size_t)s * a.M * a.nout + at;
          if (al && c + 4 <= left) {
            *(f32x4*)dst = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (c + i < left) dst[i] = v[i];
          }
        } else if (al && c + 4 <= left) {
          *(u32x2*)(a.y + at) = u32x2{pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3])};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (c + i < left) a.y[at + i] = f2bf(v[i]);
        }
      }
  };

  // ---- the stream ----
  aim();
  for (int i = 0; i < Z::NST - 1 && ui < u1; ++i) issue();
  // A wave's loads land in issue order, so the count of its later loads covers the stage; stores in
  // between only make it wait for more.
  int slot = 0, uend = unit_of(a, chunk + 1);                          // end of the current chunk
  for (int u = u0; u < u1; ++u) {
    const int rem = min(Z::NST - 2, u1 - 1 - u);                       // stages requested after this one
    if (ni == Z::IPW) wait_stages<Z::NST - 2, Z::IPW>(rem);
    else wait_stages<Z::NST - 2, Z::IPW - 1>(rem);
    lds_barrier();
    if (ui < u1) issue();
    const unsigned char* st = smem + slot * Z::STAGE;
    u32x4 wf[Z::NTW], xf[BMT];
#pragma unroll
    for (int n = 0; n < Z::NTW; ++n) wf[n] = *(const u32x4*)(st + frag(min(nt_of(n), NT - 1) * 16 + l16));
#pragma unroll
    for (int m = 0; m < BMT; ++m) xf[m] = *(const u32x4*)(st + Z::STAGE_W + frag(m * 16 + l16));
#pragma unroll
    for (int n = 0; n < Z::NTW; ++n)
#pragma unroll
      for (int m = 0; m < BMT; ++m) acc[n][m] = mfma16x16x32(wf[n], xf[m], acc[n][m]);
    const int cur = slot;
    slot = slot + 1 == Z::NST ? 0 : slot + 1;
    if (u + 1 < uend) continue;
    // end of the chunk: add the k-slices (in order) in the slice-0 waves,
    // through the stage just consumed (it is requested into again after the next stage's barrier)
    f32x4* red = (f32x4*)(smem + cur * Z::STAGE) + lane;
#pragma unroll
    for (int p = 0; p < Z::PASSES; ++p) {
      const int m0 = p * Z::RTILES, m1 = m0 + Z::RTILES < BMT ? m0 + Z::RTILES : BMT;
      lds_barrier();
      if (kslice > 0) {
#pragma unroll
        for (int n = 0; n < Z::NTW; ++n)
#pragma unroll
          for (int m = m0; m < m1; ++m) red[(((kslice - 1) * Z::NG * Z::NTW + nt_of(n)) * Z::RTILES + m - m0) * 64] = acc[n][m];
      }
      lds_barrier();
      if (kslice == 0) {
#pragma unroll
        for (int n = 0; n < Z::NTW; ++n)
#pragma unroll
          for (int m = m0; m < m1; ++m) {
            f32x4 t[Z::KW - 1];
#pragma unroll
            for (int s = 0; s < Z::KW - 1; ++s) t[s] = red[((s * Z::NG * Z::NTW + nt_of(n)) * Z::RTILES + m - m0) * 64];
#pragma unroll
            for (int s = 0; s < Z::KW - 1; ++s) acc[n][m] += t[s];
          }
      }
    }
    finish(chunk / a.S, chunk % a.S);
    clear();
    uend = unit_of(a, ++chunk + 1);
  }
}

}  // namespace lin
}  // namespace dd

// ------------------------------------------------------------------------------------------
// C ABI
#include "api.h"

using namespace dd;

namespace {

struct Plan {
  int bmt, nt, nv, nout, KT, S, C, G;
  size_t ws_bytes;
};

// The tiling of one product. N: rows of W (mode SILU: 2 I). Returns false for shapes not taken.
bool plan_for(int mode, int M, int N, int K, Plan& p) {
  if (M < 1 || M > (mode == lin::OUT ? 64 : mode == lin::SILU ? 96 : 128) || N < 1 || K < 64 || K % 64 != 0) return false;
  if ((long long)N * K >= (1ll << 30) || (long long)M * K >= (1ll << 30)) return false;   // buffer offsets
  if (mode == lin::SILU && N % 2 != 0) return false;
  const int G = cu_count();
  if (G <= 0) return false;
  p.nout = mode == lin::SILU ? N / 2 : N;
  p.bmt = (M + 15) / 16;
  if (p.bmt > 4) p.bmt += p.bmt & 1;                                   // 6, 8: rows past M cost no loads
  const int per16 = mode == lin::SILU ? 8 : 16;                        // outputs of a 16-row weight tile
  // S: parts of K (PART: the sums meet in the norm's launch); nv: outputs of S workgroups, in tiles of at
  // most 128 rows
  int nv = 0;
  for (p.S = 1;; p.S *= 2) {
    nv = (int)(((long long)p.nout * p.S + G - 1) / G);
    if (mode != lin::PART || p.S == 8 || M <= 4 * nv) break;
  }
  const int parts = (nv + 8 * per16 - 1) / (8 * per16);
  p.nv = nv = (nv + parts - 1) / parts;
  // weight tiles a stage: the narrow stages are deeper, so that they hold as many bytes. (The sums reach 5
  // and 8 only with fewer CUs than a whole card's 256, as in its compute partitions: N <= 4096.)
  const int tiles16 = (nv + per16 - 1) / per16;
  p.nt = tiles16 == 1 && p.bmt <= 2 && K % 256 == 0 ? 1
       : tiles16 <= 2 && K % 128 == 0               ? 2
       : tiles16 <= 4                               ? 4
       : tiles16 == 5                               ? 5
                                                    : 8;
  p.KT = K / (p.nt == 1 ? 256 : p.nt == 2 ? 128 : 64);
  if (p.S > p.KT) p.S = p.KT;
  const int ntiles = (p.nout + nv - 1) / nv;
  if ((long long)ntiles * p.KT >= (1ll << 30)) return false;
  p.C = ntiles * p.S;
  p.G = p.C < G ? p.C : G;
  p.ws_bytes = mode == lin::PART ? (size_t)p.S * M * N * 4 : 16;
  return true;
}

template <int BMT, int NT, int MODE>
int launch1(const lin::Args& a, int G, hipStream_t stream) {
  using Z = lin::Geo<BMT, NT>;
  auto kern = lin::linear_kernel<BMT, NT, MODE>;
  static std::atomic<unsigned long long> done;
  const hipError_t e = allow_lds((const void*)kern, Z::LDS, done);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kern, dim3(G), dim3(lin::THREADS), Z::LDS, stream, a);
  return launch_status();
}

template <int BMT, int MODE>
int launch_nt(const lin::Args& a, const Plan& p, hipStream_t stream) {
  if constexpr (BMT <= 2)
    if (p.nt == 1) return launch1<BMT, 1, MODE>(a, p.G, stream);
  if (p.nt == 2) return launch1<BMT, 2, MODE>(a, p.G, stream);
  if (p.nt == 4) return launch1<BMT, 4, MODE>(a, p.G, stream);
  if (p.nt == 5) return launch1<BMT, 5, MODE>(a, p.G, stream);
  return launch1<BMT, 8, MODE>(a, p.G, stream);
}

template <int MODE>
int launch(const Plan& p, const void* x, const void* W, void* y, int M, int N, int K, void* ws, hipStream_t stream) {
  lin::Args a;
  a.x = (const bf16*)x;
  a.W = (const bf16*)W;
  a.y = (bf16*)y;
  a.ws = (float*)ws;
  a.M = M;
  a.N = N;
  a.K = K;
  a.nout = p.nout;
  a.nv = p.nv;
  a.KT = p.KT;
  a.S = p.S;
  a.C = p.C;
  switch (p.bmt) {
    case 1: return launch_nt<1, MODE>(a, p, stream);
    case 2: return launch_nt<2, MODE>(a, p, stream);
    case 3: return launch_nt<3, MODE>(a, p, stream);
    case 4: return launch_nt<4, MODE>(a, p, stream);
  }
  if constexpr (MODE != lin::OUT)
    if (p.bmt == 6) return launch_nt<6, MODE>(a, p, stream);
  if constexpr (MODE == lin::PART) return launch_nt<8, MODE>(a, p, stream);
  return (int)hipErrorInvalidValue;
}

}  // namespace

DD_API int dd_linear_supported(int M, int N, int K) {
  Plan p;
  return plan_for(lin::OUT, M, N, K, p) ? 1 : 0;
}

DD_API size_t dd_linear_add_rmsnorm_ws_bytes(int M, int N, int K) {
  Plan p;
  return plan_for(lin::PART, M, N, K, p) ? p.ws_bytes : 0;
}

DD_API int dd_linear(const void* x, const void* W, void* y, int M, int N, int K, hipStream_t stream) {
  Plan p;
  DD_REQUIRE(x && W && y && plan_for(lin::OUT, M, N, K, p));
  DD_REQUIRE(aligned16(x) && aligned16(W) && aligned16(y));
  return launch<lin::OUT>(p, x, W, y, M, N, K, nullptr, stream);
}

DD_API int dd_linear_silu(const void* x, const void* Wgu, void* out, int M, int I, int K, hipStream_t stream) {
  Plan p;
  DD_REQUIRE(x && Wgu && out && I >= 1 && I < (1 << 30) && plan_for(lin::SILU, M, 2 * I, K, p));
  DD_REQUIRE(aligned16(x) && aligned16(Wgu) && aligned16(out));
  return launch<lin::SILU>(p, x, Wgu, out, M, 2 * I, K, nullptr, stream);
}

DD_API int dd_linear_add_rmsnorm(const void* x, const void* W, const void* h, const void* lnw, void* hn, void* y,
                                 int M, int N, int K, float eps, void* ws, hipStream_t stream) {
  Plan p;
  DD_REQUIRE(x && W && h && lnw && hn && y && ws && N <= 4096 && plan_for(lin::PART, M, N, K, p));
  DD_REQUIRE(aligned16(x) && aligned16(W) && aligned16(ws));
  const int rc = launch<lin::PART>(p, x, W, nullptr, M, N, K, ws, stream);
  return rc != 0 ? rc : launch_sum_add_rmsnorm(ws, p.S, h, lnw, hn, y, M, N, eps, stream);
}
