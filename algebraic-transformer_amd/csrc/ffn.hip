// ALU-GLU feed-forward for gfx950: the activation and its VJP fused into the epilogues of the
// products that produce and consume it (src/algebraic/model.py:185-193, ffn = "alu_glu";
// alu and its custom VJP: src/algebraic/algebraic.py:86-113).
//
// Forward: [gate | up] = h2 [w_g | w_u] as one product over the concatenated weights (a split
// operand: each wave's two 32-column blocks are the same columns f of w_g and of w_u), and the
// epilogue forms gate = round(.), up = round(.), act = alu(up), y = round(gate act); it stores
// y for the output product and gate, up for the backward.
// Backward: dy = round(dout w_d^T) with the epilogue forming d_gate = round(dy act),
// d_act = round(dy gate), d_up = round(d_act (0.5 (1 + u) + 0.5 u r^2)) (u, r recomputed from
// up), stored as one (N, 2F) matrix [d_gate | d_up] so dh2 and [dw_g | dw_u] are one product
// each. The remaining products (y w_d, dh2, the weight gradients) are plain GEMMs.
#include <algorithm>
#include <cmath>

#include "gemm_core.h"
#include "head_params.h"
#include "launchers.h"

#pragma clang fp contract(off)

namespace alg {

typedef HeadGemm FC;                    // 256 x 256 tiles, 8 waves (2 x 4)
typedef GemmCfg<128, 128, 2, 2> FC128;  // products that fill less of the chip
typedef GemmCfg<64, 64, 2, 2> FC64;

namespace {

// alu(z) with the reference's negative-tail form; u, r returned for the derivative
// (algebraic.py:84-91). r is the hardware reciprocal square root, as the reference's
// lax.rsqrt; the tail's r^2 / (1 - u) (1 - u in (1, 2)) is a reciprocal multiply, within
// 2 ulp of the f32 quotient before the result is rounded to bf16. An IEEE sqrt and two IEEE
// divisions here cost about three times the VALU of the rest of the epilogue.
__device__ __forceinline__ float alu_f32(float z, float beta, float& u, float& r) {
  const float bz = __fmul_rn(beta, z);
  r = rsq(__fadd_rn(1.0f, __fmul_rn(bz, bz)));
  u = __fmul_rn(bz, r);
  const float one_plus_u =
      bz < 0.0f ? __fmul_rn(__fmul_rn(r, r), __builtin_amdgcn_rcpf(__fsub_rn(1.0f, u))) : __fadd_rn(1.0f, u);
  return __fmul_rn(__fmul_rn(0.5f, z), one_plus_u);
}

__device__ __forceinline__ float rb(float x) { return (float)f2bf(x); }

// Each wave stages its WTM x WTN block of bf16 values in its own share of the (idle) pipeline
// buffers, rows of WTN / 8 16-byte chunks XOR-swizzled by the row, so the accumulator's
// column-per-lane writes spread over the banks and the 16-byte row reads stay aligned; the
// global loads and stores of the epilogue then move 8 consecutive columns per lane.
template <int W>
__device__ __forceinline__ int stage_at(int r, int c) {
  return r * W + (((c >> 3) ^ (r & (W / 8 - 1))) << 3) + (c & 7);
}

// Tile (m0, n0) of A B over k in [kbeg, kend), handed to epi(acc, stage) with this wave's
// staging share, free of readers.
template <int AM, int BM, class C, class Epi>
__device__ __forceinline__ void ffn_tile(const GemmOperand& A, const GemmOperand& B, int m0, int n0, int kbeg, int kend,
                                         Epi epi) {
  static_assert(gemm_share<AM, BM, C>() >= C::WTM * C::WTN, "a wave's block fits its share");
  floatx16 acc[C::MB][C::NB];
  bf16* stage = gemm_tile<AM, BM, C>(A, B, m0, n0, kbeg, kend, acc);
  __syncthreads();  // every wave is done reading the pipeline buffers
  epi(acc, stage);
}

}  // namespace

// The weights in bf16, [w_g | w_u] side by side: one pass in place of a concatenation, its
// conversion and w_d's (bound by memory; f32 weights of d 768, d_ff 2048: 17 us of three kernels,
// 7 us so).
__global__ __launch_bounds__(256) void ffn_pack_kernel(FfnPackParams p) {
  const int n1 = p.d * (p.F / 8), n2 = p.w_d16 ? p.F * (p.dm / 8) : 0;  // 8-element chunks
  for (int i = blockIdx.x * 256 + threadIdx.x; i < 2 * n1 + n2; i += gridDim.x * 256) {
    const int part = i < n1 ? 0 : i < 2 * n1 ? 1 : 2;
    const int c = i - part * n1;
    const void* src = part == 0 ? p.w_g : part == 1 ? p.w_u : p.w_d;
    bf16x8 v;
    if (part == 0 ? p.g_f32 : part == 1 ? p.u_f32 : p.d_f32) {
      const floatx4 x = static_cast<const floatx4*>(src)[2 * (size_t)c], y = static_cast<const floatx4*>(src)[2 * (size_t)c + 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = f2bf(x[e]);
        v[4 + e] = f2bf(y[e]);
      }
    } else {
      v = static_cast<const bf16x8*>(src)[c];
    }
    const int row = c / (p.F / 8);
    bf16* dst = part == 2 ? p.w_d16 + 8 * (size_t)c
                          : p.w_gu + (size_t)row * 2 * p.F + part * p.F + 8 * (c - row * (p.F / 8));
    *reinterpret_cast<bf16x8*>(dst) = v;
  }
}

template <class C>
__global__ __launch_bounds__(C::THREADS, 2) void ffn_gate_up_kernel(FfnParams p) {
  const int nbm = (p.N + C::TM - 1) / C::TM, nbn = 2 * p.F / C::TN;
  int tm, tn;
  xcd_tile(blockIdx.x, nbm, nbn, tm, tn);
  const int m0 = tm * C::TM, n0 = tn * C::TN;  // tokens, logical [gate | up] columns
  GemmOperand A{p.h2, p.d, p.N, p.d, (long)p.N * p.d};
  GemmOperand B{p.w_gu, 2L * p.F, p.d, 2 * p.F, 2L * p.d * p.F, (long)p.F};
  ffn_tile<KMAJOR, MNMAJOR, C>(A, B, m0, n0, 0, p.d, [&](const floatx16 (&acc)[C::MB][C::NB], bf16* stg) {
    static_assert(C::NB == 2, "a wave's two column blocks are gate and up");
    const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
    int wm, wn;
    wave_coords<C>(wm, wn);
    // acc[.][0] is gate column f0 + l32, acc[.][1] up column f0 + l32 (f0 = n0/2 + 32 wn);
    // staged as [row][0..31] gate, [row][32..63] up.
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
        stg[stage_at<64>(row, l32)] = f2bf(acc[mb][0][i]);
        stg[stage_at<64>(row, 32 + l32)] = f2bf(acc[mb][1][i]);
      }
    }
    // WTM rows x 4 chunks of 8 columns: lane -> (row, chunk).
    const int f0 = n0 / 2 + wn * 32;
#pragma unroll
    for (int it = 0; it < C::WTM / 16; ++it) {
      const int idx = it * 64 + lane, row = idx >> 2, ch = idx & 3;
      const int tok = m0 + wm * C::WTM + row;
      const bf16x8 gv = *reinterpret_cast<const bf16x8*>(stg + stage_at<64>(row, 8 * ch));
      const bf16x8 uv = *reinterpret_cast<const bf16x8*>(stg + stage_at<64>(row, 32 + 8 * ch));
      bf16x8 yv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float u, r;
        const float act = rb(alu_f32((float)uv[e], p.beta, u, r));
        yv[e] = f2bf(__fmul_rn((float)gv[e], act));
      }
      if (tok < p.N) {
        const size_t o = (size_t)tok * p.F + f0 + 8 * ch;
        *reinterpret_cast<bf16x8*>(p.y + o) = yv;
        *reinterpret_cast<bf16x8*>(p.gate + o) = gv;
        *reinterpret_cast<bf16x8*>(p.up + o) = uv;
      }
    }
  });
}

template <class C>
__global__ __launch_bounds__(C::THREADS, 2) void ffn_dy_kernel(FfnParams p) {
  const int nbm = (p.N + C::TM - 1) / C::TM, nbn = (p.F + C::TN - 1) / C::TN;
  int tm, tn;
  xcd_tile(blockIdx.x, nbm, nbn, tm, tn);
  const int m0 = tm * C::TM, n0 = tn * C::TN;  // tokens, columns f
  GemmOperand A{p.dout, p.dm, p.N, p.dm, (long)p.N * p.dm};
  GemmOperand B{p.w_d, p.dm, p.F, p.dm, (long)p.F * p.dm};  // w_d (F, dm): [f][k]
  ffn_tile<KMAJOR, KMAJOR, C>(A, B, m0, n0, 0, p.dm, [&](const floatx16 (&acc)[C::MB][C::NB], bf16* stg) {
    constexpr int W = C::WTN, CH = W / 8;  // this wave's dy block, [row][0..W)
    const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
    int wm, wn;
    wave_coords<C>(wm, wn);
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) stg[stage_at<W>(row, nb * 32 + l32)] = f2bf(acc[mb][nb][i]);
      }
    }
    // WTM rows x CH chunks of 8 columns: lane -> (row, chunk), in groups of GRP chunks per lane
    // whose gate/up loads are issued together (out-of-range chunks read chunk 0 and are not
    // stored): behind a per-chunk range check each load got a branch and a wait of its own.
    const int f0 = n0 + wn * W;
    constexpr int PER = C::WTM * CH / 64, GRP = PER < 8 ? PER : 8;
#pragma unroll 1
    for (int g0 = 0; g0 < PER; g0 += GRP) {
      bf16x8 gvs[GRP], uvs[GRP];
#pragma unroll
      for (int k = 0; k < GRP; ++k) {
        const int idx = (g0 + k) * 64 + lane, row = idx / CH, ch = idx % CH;
        const int tok = m0 + wm * C::WTM + row, f = f0 + 8 * ch;
        const size_t o = tok < p.N && f < p.F ? (size_t)tok * p.F + f : 0;
        gvs[k] = *reinterpret_cast<const bf16x8*>(p.gate + o);
        uvs[k] = *reinterpret_cast<const bf16x8*>(p.up + o);
      }
#pragma unroll
      for (int k = 0; k < GRP; ++k) asm volatile("" : "+v"(gvs[k]), "+v"(uvs[k]));  // loads before the checks
#pragma unroll
      for (int k = 0; k < GRP; ++k) {
        const int idx = (g0 + k) * 64 + lane, row = idx / CH, ch = idx % CH;
        const int tok = m0 + wm * C::WTM + row, f = f0 + 8 * ch;
        if (tok >= p.N || f >= p.F) continue;  // F is a multiple of 128: chunks are whole
        const bf16x8 dyv = *reinterpret_cast<const bf16x8*>(stg + stage_at<W>(row, 8 * ch));
        const bf16x8 gv = gvs[k], uv = uvs[k];
        bf16x8 dg, du;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float dy = (float)dyv[e];
          float u, r;
          const float act = rb(alu_f32((float)uv[e], p.beta, u, r));
          const float d_act = rb(__fmul_rn(dy, (float)gv[e]));
          const float deriv =
              __fadd_rn(__fmul_rn(0.5f, __fadd_rn(1.0f, u)), __fmul_rn(__fmul_rn(0.5f, u), __fmul_rn(r, r)));
          dg[e] = f2bf(__fmul_rn(dy, act));
          du[e] = f2bf(__fmul_rn(d_act, deriv));
        }
        const size_t od = (size_t)tok * 2 * p.F + f;
        *reinterpret_cast<bf16x8*>(p.d_gu + od) = dg;
        *reinterpret_cast<bf16x8*>(p.d_gu + od + p.F) = du;
      }
    }
  });
}

// Plain products of the block (model.py:185-193: y w_d in the forward; [d_gate | d_up] [w_g |
// w_u]^T, h2^T [d_gate | d_up] and y^T dout in the backward): C = A B, one rounding to bf16 of
// the f32 sum, each operand read in its stored layout (AM, BM), so no transposed copy is made.
// Workgroups below g.full compute whole tiles, row-major inside each XCD's share; the rest
// compute k range (id - full) % split of tile full + (id - full) / split into an f32 tile of
// g.part, which ffn_gemm_tail_kernel sums in range order (ffn_gemm_plan).
template <int AM, int BM, class C>
__global__ __launch_bounds__(C::THREADS, 2) void ffn_gemm_kernel(FfnGemmParams g) {
  const int nbn = (g.N + C::TN - 1) / C::TN;
  const int bid = blockIdx.x;
  int lin, kbeg = 0, kend = g.K, unit = -1;
  if (bid < g.full) {
    // A share of rows per XCD reads all of B on every XCD. Where B is the larger operand and the row
    // length lets the plain order give an XCD every fourth column, or fewer, that is the better one
    // (M N K 1600 3328 1536: 44 us in shares, 33 plain; 704 5888 2115: 45 / 37).
    lin = g.full % 8 && nbn % 4 == 0 && g.N > g.M ? bid : xcd_contiguous(bid, g.full);
  } else {
    unit = bid - g.full;
    lin = g.full + unit / g.split;
    kbeg = (unit % g.split) * g.kchunk;
    kend = min(g.K, kbeg + g.kchunk);
  }
  const int tm = lin / nbn, tn = lin - tm * nbn;
  const int m0 = tm * C::TM, n0 = tn * C::TN;
  ffn_tile<AM, BM, C>(g.A, g.B, m0, n0, kbeg, kend, [&](const floatx16 (&acc)[C::MB][C::NB], bf16* stg) {
    constexpr int W = C::WTN, CH = W / 8;
    const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
    int wm, wn;
    wave_coords<C>(wm, wn);
    if (unit >= 0) {  // one k range of a split tile: the whole f32 tile, row-major
      float* part = g.part + (size_t)unit * C::TM * C::TN;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int r = wm * C::WTM + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
#pragma unroll
          for (int nb = 0; nb < C::NB; ++nb) part[r * C::TN + wn * W + nb * 32 + l32] = acc[mb][nb][i];
        }
      return;
    }
    // n2 is a multiple of 64, so a wave's columns lie on one side of it.
    const int mw = m0 + wm * C::WTM, nw = n0 + wn * W;
    const bool second = nw >= g.n2;
    const int nc = second ? nw - g.n2 : nw, ncols = second ? g.N - g.n2 : g.n2;
    void* base = second ? g.C2 : g.C;
    if (second ? g.c2_f32 : g.c_f32) {
      float* out = static_cast<float*>(base) + (size_t)mw * g.ldc + nc;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int row = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
#pragma unroll
          for (int nb = 0; nb < C::NB; ++nb)
            if (mw + row < g.M && nc + nb * 32 + l32 < ncols) out[(size_t)row * g.ldc + nb * 32 + l32] = acc[mb][nb][i];
        }
      }
      return;
    }
    // Staged 16-byte row stores; N is a multiple of 8, so a chunk lies inside a row or past it.
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) stg[stage_at<W>(row, nb * 32 + l32)] = f2bf(acc[mb][nb][i]);
      }
    }
    bf16* out = static_cast<bf16*>(base) + (size_t)mw * g.ldc + nc;
    const bool inside = m0 + C::TM <= g.M && n0 + C::TN <= g.N;
#pragma unroll 4
    for (int it = 0; it < C::WTM * CH / 64; ++it) {
      const int idx = it * 64 + lane, row = idx / CH, ch = idx % CH;
      if (inside || (mw + row < g.M && nc + 8 * ch < ncols))
        *reinterpret_cast<bf16x8*>(out + (size_t)row * g.ldc + 8 * ch) =
            *reinterpret_cast<const bf16x8*>(stg + stage_at<W>(row, 8 * ch));
    }
  });
}

// C of a split tile: its split f32 range tiles summed in range order, 32 rows of the tile per
// workgroup (grid: split tiles x TM / 32). N is a multiple of 8, so 8 columns that start
// inside the matrix lie inside it.
template <class C>
__global__ __launch_bounds__(256) void ffn_gemm_tail_kernel(FfnGemmParams g) {
  const int nbn = (g.N + C::TN - 1) / C::TN;
  const int lin = g.full + blockIdx.x;
  const int tm = lin / nbn, tn = lin - tm * nbn;
  const float* part = g.part + (size_t)blockIdx.x * g.split * C::TM * C::TN;
#pragma unroll
  for (int c = 0; c < 32 * C::TN / 8 / 256; ++c) {
    const int e = (threadIdx.x + 256 * c) * 8;
    const int r = blockIdx.y * 32 + e / C::TN, col = e % C::TN;
    const int m = tm * C::TM + r, n = tn * C::TN + col;
    if (m >= g.M || n >= g.N) continue;
    const size_t o = (size_t)r * C::TN + col;
    float4 a = *reinterpret_cast<const float4*>(part + o), b = *reinterpret_cast<const float4*>(part + o + 4);
    for (int k = 1; k < g.split; ++k) {
      const float* q = part + (size_t)k * C::TM * C::TN + o;
      const float4 x = *reinterpret_cast<const float4*>(q), y = *reinterpret_cast<const float4*>(q + 4);
      a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      b.x += y.x; b.y += y.y; b.z += y.z; b.w += y.w;
    }
    const bool second = n >= g.n2;
    const size_t at = (size_t)m * g.ldc + (second ? n - g.n2 : n);
    void* base = second ? g.C2 : g.C;
    if (second ? g.c2_f32 : g.c_f32) {
      float4* out = reinterpret_cast<float4*>(static_cast<float*>(base) + at);
      out[0] = a;
      out[1] = b;
      continue;
    }
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    bf16x8 o8;
#pragma unroll
    for (int t = 0; t < 8; ++t) o8[t] = f2bf(v[t]);
    *reinterpret_cast<bf16x8*>(static_cast<bf16*>(base) + at) = o8;
  }
}

static int ffn_tiles(int tile, int M, int N) { return ((M + tile - 1) / tile) * ((N + tile - 1) / tile); }

// Tile of the gate/up product: 128 where its tiles run in one round of the CUs, or, when no tile is
// ragged in the tokens, in two, or in more when gemm_tile_time says so. Its weights come in 64-byte pieces (gate and up columns alternate), so
// later rounds of 128 tiles, and ragged ones above all, cost more than those of 256 (N d F, us,
// 256 / 128; 2048 512 1408: 22.0 / 20.4; 1000 1024 2816: 36 / 40; 400 2048 5632: 57 / 89;
// 3500 1024 2816: 67 / 120; 6528 960 1280: 64 / 52).
int ffn_gate_up_tile(int N, int F, int d) {
  const int tiles = ffn_tiles(128, N, 2 * F);
  if (tiles <= 256) return 128;
  if (N % 128) return 256;
  return tiles <= 512 || gemm_tile_time(128, tiles, d, N, 2 * F) <
                             gemm_tile_time(256, ffn_tiles(256, N, 2 * F), d, N, 2 * F) ? 128 : 256;
}

// Tile of the dout w_d^T product with the activation's VJP: 64 while gemm_tile_time says so. The
// epilogue reads gate and up and writes their gradients, 9.9 us a round of 256 tiles, where two
// workgroups of 64 tiles to a CU hide each other's (N dm F, us, 256 / 128 / 64; 1500 1024 2816:
// 41.6 / 46.8 / 27.7; 2500 768 2048: 36.2 / 39.2 / 25.3; 4096 1024 2816: 43.7 / 54.1 / 47.3; 128 tiles
// were the best nowhere by more than 0.6 us).
int ffn_dy_tile(int N, int F, int dm) {
  const int t256 = ffn_tiles(256, N, F), rounds = (t256 + 255) / 256;
  return gemm_tile_time(64, ffn_tiles(64, N, F), dm, N, F) < gemm_tile_time(256, t256, dm, N, F) + 9.9 * rounds ? 64 : 256;
}

// Plan of a plain product. With 256 x 256 tiles, those past the last complete round of 256
// workgroups (all of them when there are fewer than 256) are split over k into S ranges when that
// is cheaper. Cost model, from the head products' measured rates: a round of 256 x 256 tiles
// costs 23.4 ns per k step of one element (48 us for K = 2048), and each split range tile costs
// its f32 tile written, read and summed (512 KiB at about 5 TB/s over the chip, 0.1 us) plus 5 us
// for the summing launch. A range keeps at least 1024 of K (so every range is non-empty). The
// workspace is that of this split. A product that fills less of the chip runs on smaller tiles
// when gemm_tile_time says so (a split: 3 us for its summing launch and its f32 tiles written and
// read at 15 TB/s, out of the caches); 64 x 64 tiles are split over k (ranges of at least 512) as
// far as the same workspace goes, which pays where few tiles have a long k (304 1024 4096: 26.9 us
// whole, 15.0 us in four ranges).
FfnGemmPlan ffn_gemm_plan(int M, int N, int K) {
  FfnGemmPlan pl;
  pl.tile = 256;
  pl.tiles = ffn_tiles(256, M, N);
  pl.full = pl.tiles;
  pl.split = 1;
  pl.kchunk = 0;
  pl.ws_bytes = 0;
  const int base = pl.tiles / 256 * 256, tail = pl.tiles - base;
  if (tail) {
    auto cost = [&](int s) {
      const double rounds = std::ceil(tail * (double)s / 256.0);
      return rounds * (K / (double)s) * 0.0234 + (s > 1 ? tail * s * 0.1 + 5.0 : 0.0);
    };
    int best = 1;
    double best_cost = cost(1);
    for (int s = 2; s <= 8 && K / s >= 1024; ++s) {
      const double c = cost(s);
      if (c < best_cost - 1e-9) { best = s; best_cost = c; }
    }
    if (best > 1) {
      pl.full = base;
      pl.split = best;
      pl.kchunk = ((K + best - 1) / best + 127) / 128 * 128;
      pl.ws_bytes = (size_t)tail * best * 256 * 256 * sizeof(float);
    }
  }
  if (base) return pl;  // a whole round of 256 tiles: the chip is full
  auto time = [&](int tile, int units, int s, int chunk) {
    return gemm_tile_time(tile, units, chunk, M, N) + (s > 1 ? 3.0 + 8e-6 * 0.067 * units * tile * tile : 0.0);
  };
  double best_time = time(256, pl.tiles * pl.split, pl.split, pl.split == 1 ? K : pl.kchunk);
  auto consider = [&](int tile, int s) {
    const int tiles = ffn_tiles(tile, M, N);
    const int chunk = s > 1 ? ((K + s - 1) / s + 127) / 128 * 128 : K;
    const double t = time(tile, tiles * s, s, chunk);
    if (t >= best_time) return;
    best_time = t;
    pl.tile = tile;
    pl.tiles = tiles;
    pl.full = s > 1 ? 0 : tiles;
    pl.split = s;
    pl.kchunk = s > 1 ? chunk : 0;
  };
  consider(128, 1);
  consider(64, 1);
  const size_t plane = (size_t)ffn_tiles(64, M, N) * 64 * 64 * sizeof(float);
  for (int s = 2; s <= 8 && K / s >= 512 && s * plane <= pl.ws_bytes; s *= 2) consider(64, s);
  return pl;
}

template <class C>
static void launch_ffn_gemm_cfg(const FfnGemmParams& g, int a_mode, int b_mode, hipStream_t st) {
  const int tiles = ((g.M + C::TM - 1) / C::TM) * ((g.N + C::TN - 1) / C::TN);
  const dim3 grid(g.split > 1 ? g.full + (tiles - g.full) * g.split : tiles), nt(C::THREADS);
  {
    KTimer t("ffn_gemm", st);
    if (a_mode == KMAJOR && b_mode == KMAJOR) hipLaunchKernelGGL((ffn_gemm_kernel<KMAJOR, KMAJOR, C>), grid, nt, 0, st, g);
    else if (a_mode == KMAJOR) hipLaunchKernelGGL((ffn_gemm_kernel<KMAJOR, MNMAJOR, C>), grid, nt, 0, st, g);
    else if (b_mode == KMAJOR) hipLaunchKernelGGL((ffn_gemm_kernel<MNMAJOR, KMAJOR, C>), grid, nt, 0, st, g);
    else hipLaunchKernelGGL((ffn_gemm_kernel<MNMAJOR, MNMAJOR, C>), grid, nt, 0, st, g);
  }
  if (g.split > 1) {
    KTimer t("ffn_gemm_tail", st);
    hipLaunchKernelGGL(ffn_gemm_tail_kernel<C>, dim3(tiles - g.full, C::TM / 32), dim3(256), 0, st, g);
  }
}

hipError_t launch_ffn_gemm(const FfnGemmParams& g, int a_mode, int b_mode, hipStream_t st) {
  if (g.tile == 64) launch_ffn_gemm_cfg<FC64>(g, a_mode, b_mode, st);
  else if (g.tile == 128) launch_ffn_gemm_cfg<FC128>(g, a_mode, b_mode, st);
  else launch_ffn_gemm_cfg<FC>(g, a_mode, b_mode, st);
  return hipGetLastError();
}

hipError_t launch_ffn_pack(const FfnPackParams& p, hipStream_t st) {
  const long chunks = 2L * p.d * (p.F / 8) + (p.w_d16 ? (long)p.F * (p.dm / 8) : 0);
  KTimer t("ffn_pack", st);
  hipLaunchKernelGGL(ffn_pack_kernel, dim3((int)std::min(2048L, (chunks + 255) / 256)), dim3(256), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_ffn_fwd(const FfnParams& p, hipStream_t st) {
  KTimer t("ffn_gate_up", st);
  if (ffn_gate_up_tile(p.N, p.F, p.d) == 128)
    hipLaunchKernelGGL(ffn_gate_up_kernel<FC128>, dim3(ffn_tiles(128, p.N, 2 * p.F)), dim3(FC128::THREADS), 0, st, p);
  else
    hipLaunchKernelGGL(ffn_gate_up_kernel<FC>, dim3(ffn_tiles(256, p.N, 2 * p.F)), dim3(FC::THREADS), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_ffn_dy(const FfnParams& p, hipStream_t st) {
  KTimer t("ffn_dy", st);
  const int tile = ffn_dy_tile(p.N, p.F, p.dm);
  const dim3 grid(ffn_tiles(tile, p.N, p.F));
  if (tile == 64) hipLaunchKernelGGL(ffn_dy_kernel<FC64>, grid, dim3(FC64::THREADS), 0, st, p);
  else hipLaunchKernelGGL(ffn_dy_kernel<FC>, grid, dim3(FC::THREADS), 0, st, p);
  return hipGetLastError();
}

}  // namespace alg
