// Fused tied-embedding algebraic likelihood head for gfx950.
//
// Replaces src/algebraic/kernels/fused_head.py:72-275 (forward statistics, telemetry,
// backward) including the XLA embedding-gradient matmul of fused_head.py:215.
//
// Forward (logits never stored): z^T = E h^T per 256 vocab x 256 token tile (bf16 MFMA, f32
// accumulate); the epilogue forms x = min(z/c, X), w = rho_fast(x)^n, r = rsqrt(1+x^2),
// per-token partial sums of w for this vocab tile and the target logit zt
// (fused_head.py:83-103). A statistics kernel reduces the partials in a fixed order:
// stat = l^(-1/n) (fused_head.py:116), telemetry pt = (rho(min(zt/c, X)) stat)^n and the
// objective mean(1 - pt) (fused_head.py:219-229).
//
// Backward, three schedules over the same GEMM core:
//  * residual (3 products): with p = w/l the logit gradient is
//        dz = s (p - y) r = (s/l) U',  U' = w r except U'_t = (w_t - l) r_t,
//    so the forward epilogue also stores U = bf16(w r) token-major and the statistics kernel
//    patches the target entries once l is known. Then dh = (s/l) (U' E) and
//    dE = U'^T (s h / l): no logit recompute.
//  * recompute (4 products, the reference's schedule, fused_head.py:120-156, 194-216): the
//    backward recomputes z, writes bf16(s (p - y) r) token-major, then dh = dZ E and
//    dE = dZ^T h.
//  * streamed (the recompute schedule one vocabulary chunk at a time, launch_head_bwd_streamed):
//    per chunk dZ of the chunk only, its dh product accumulated in f32 across the chunks and its
//    rows of dE, so no (N, V) block is held at all.
// Every product reads its operands in their natural layout (k-contiguous fragments via
// ds_read_b128, transposed ones via ds_read_b64_tr_b16).
#include <cmath>
#include <type_traits>

#include "gemm_core.h"
#include "head_eval.h"
#include "head_params.h"
#include "launchers.h"

namespace alg {

typedef HeadGemm HC;                    // 256 x 256 tiles, 8 waves (2 x 4)
typedef GemmCfg<128, 128, 2, 2> HC128;  // products that fill less of the chip
template <class C>
constexpr int head_waves_per_simd() { return C::THREADS == 512 ? 1 : 2; }

__device__ __forceinline__ float head_w(float z, const HeadParams& p, float& r) {
  const float x = fminf(z * p.inv_c, p.clamp);  // fused_head.py:98
  float t = rho_fast(x, r);
  for (int e = 0; e < p.log2n; ++e) t = t * t;
  return t;
}

// Token-major staging of a wave's WTM (v) x WTN (tok) block of a bf16 (tok, v) matrix (the
// forward's residual U, the recompute schedules' logit gradient dZ): the wave writes its block
// into its own share of the idle pipeline buffers as [tok][v] rows, 16-byte chunks
// XOR-swizzled by the token, then stores it with 16-byte stores that cover whole token rows
// (full cache lines) per instruction.
template <class C>
__device__ __forceinline__ int ustage_at(int tl, int vl) {
  constexpr int UCH = C::WTM / 8;  // 16-byte chunks per staged token row
  static_assert(UCH <= 64 && 64 % UCH == 0 && (UCH & (UCH - 1)) == 0, "staged row width");
  return tl * C::WTM + (((vl >> 3) ^ (tl & (UCH - 1))) << 3) + (vl & 7);
}

// Stores the staged block: token rows tok0 + (0..WTN-1), vocabulary entries v0 + (0..WTM-1) of
// out (row pitch Vp, Npad rows). AUX is the store's cache policy. EDGE: chunks at or past Vp are
// dropped (Vp is a multiple of 8, so a chunk lies inside a row or past it; token rows always lie
// inside the Npad rows).
template <class C, int AUX, bool EDGE = false>
__device__ __forceinline__ void store_staged_tokmajor(const bf16* ub, bf16* out, int Npad, int Vp, int tok0, int v0,
                                                      int lane) {
  const size_t ubase = (size_t)tok0 * Vp + v0;
  const size_t rest = ((size_t)Npad * Vp - ubase) * 2;  // bytes of out from the base
  const __amdgpu_buffer_rsrc_t urs = __builtin_amdgcn_make_buffer_rsrc(
      out + ubase, (short)0, (int)std::min<size_t>(rest, 0x7fffffff), BUF_RSRC_WORD3);
  constexpr int UCH = C::WTM / 8, RPS = 64 / UCH;  // token rows per store instruction
  const int ch = lane % UCH;
  const int voff = ((lane / UCH) * Vp + ch * 8) * 2;
  // The row offset goes into the per-lane offset and the scalar offset stays the constant
  // 0. A 16-byte store needs one wait state before a VALU instruction may overwrite its
  // data registers; the compiler inserts it only when the scalar offset is not an SGPR.
  // With the row offset in an SGPR (an earlier form of this loop) the next instruction
  // reused the data registers of the store just issued, and on gfx950 the store wrote the
  // new values (measured: about 0.1 % of the U entries replaced by address arithmetic).
#pragma unroll
  for (int j = 0; j < C::WTN / RPS; ++j) {
    const int tl = RPS * j + lane / UCH;
    const u32x4 v = *reinterpret_cast<const u32x4*>(ub + ustage_at<C>(tl, ch * 8));
    if (!EDGE || v0 + ch * 8 < Vp) __builtin_amdgcn_raw_buffer_store_b128(v, urs, voff + RPS * j * Vp * 2, 0, AUX);
  }
}

// A row-major (N, d) or (V, d) operand of the head's products: bf16, or with SPLIT the three
// bf16 planes of an f32 matrix.
template <bool SPLIT>
__device__ __forceinline__ GemmOperand head_operand(const bf16* ptr, int rows, int d, long plane) {
  GemmOperand o{ptr, d, rows, d, (long)rows * d};
  if constexpr (SPLIT) o.plane = plane;
  return o;
}

// z^T = E h^T with the forward epilogue (row sums, target logit, optional U residual).
// L2N > 0 fixes n = 2^L2N at compile time (0: taken from the parameters).
// acc[mb][nb][4g + e] for the row offset dt = mb*32 + 8g + e (bit 2 of dt, the lane half,
// already matched).
template <class C>
__device__ __forceinline__ float select_row(const floatx16 (&acc)[C::MB][C::NB], int nb, int dt) {
  float z = 0.0f;
#pragma unroll
  for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) z = dt == mb * 32 + 8 * (i >> 2) + (i & 3) ? acc[mb][nb][i] : z;
  return z;
}

// SPLIT: f32 h and E as three bf16 planes each (gemm_mainloop's six passes); no residual, and
// the row sums are kept per 128 vocabulary entries, the tiling of the f32 kernels that run
// instead when a value is out of the planes' range (p.split_bad).
template <class C, int L2N, bool SPLIT>
__global__ __launch_bounds__(C::THREADS, head_waves_per_simd<C>()) void head_fwd_kernel(HeadParams p) {
  if (SPLIT && *p.split_bad) return;
  __shared__ float red[C::WM][C::TN];
  const int nbm = (p.V + C::TM - 1) / C::TM, nbn = (p.N + C::TN - 1) / C::TN;
  int tm, tn;
  xcd_tile(blockIdx.x, nbm, nbn, tm, tn);
  const int m0 = tm * C::TM;  // vocab
  const int n0 = tn * C::TN;  // tokens
  const GemmOperand A = head_operand<SPLIT>(p.E, p.V, p.d, (long)p.V * p.d);
  const GemmOperand B = head_operand<SPLIT>(p.h, p.N, p.d, (long)p.N * p.d);
  floatx16 acc[C::MB][C::NB];
  bf16* ub = gemm_tile<KMAJOR, KMAJOR, C, SPLIT>(A, B, m0, n0, 0, p.d, acc);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int wm, wn;
  wave_coords<C>(wm, wn);
  const float inv_c = p.inv_c, clamp = p.clamp;
  const int vrow0 = m0 + wm * C::WTM;  // first vocab row of this wave
  // WITH_U also stores the residual. U is token-major (element (tok, v) at tok * Vp + v),
  // staged per wave and written with 16-byte stores marked non-temporal so the 1 GB stream of U
  // does not evict the E / h panels the GEMM is reusing from L2. EDGE (tiles that reach past V
  // or N): rows past V add nothing to the sums; U's rows up to the end of the last tile and its
  // columns up to Vp are all written, as finite values wherever h is finite (operand rows past the
  // end read as zeros); nothing reads a row past N. Edge tiles once stored U an element at a time, 2 bytes a lane: at N = 1000 their
  // quarter of the tiles took most of the kernel.
  static_assert(C::WTM * C::WTN <= gemm_share<KMAJOR, KMAJOR, C>(), "a wave's block fits its share");
  auto epilogue = [&](auto with_u, auto edge) {
    constexpr bool WITH_U = decltype(with_u)::value, EDGE = decltype(edge)::value;
    if constexpr (WITH_U) __syncthreads();  // every wave is done reading the pipeline buffers
#pragma unroll
    for (int nb = 0; nb < C::NB; ++nb) {
      const int col = wn * C::WTN + nb * 32 + l32;
      const int tok = n0 + col;
      const int tgt = !EDGE || tok < p.N ? p.targets[tok] : -1;
      const int dt = tgt - vrow0 - 4 * h;  // target row relative to this lane's rows
      float part = 0.0f;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float z = acc[mb][nb][4 * g + e];
            const float x = fminf(z * inv_c, clamp);  // fused_head.py:98
            float r;
            const float w = pow2n<L2N>(rho_fast(x, r), p.log2n);
            part += !EDGE || vrow0 + mb * 32 + 8 * g + 4 * h + e < p.V ? w : 0.0f;
            u[e] = w * r;
          }
          if constexpr (WITH_U) {
            u32x2 pk;
            pk[0] = pack_bf16x2(u[0], u[1]);
            pk[1] = pack_bf16x2(u[2], u[3]);
            *reinterpret_cast<u32x2*>(ub + ustage_at<C>(nb * 32 + l32, mb * 32 + 8 * g + 4 * h)) = pk;
          }
        }
      }
      // The lane holds rows mb*32 + 8g + e (+4h) of the block: the target's row is one of them
      // when its offset dt has bit 2 clear and lies in [0, WTM). That is rare (WTM of V rows
      // per token), so the select runs behind a wave-uniform branch, skipped by every wave
      // where no lane hits. (A target past V may hit a row past V; the statistics ignore it.)
      const bool mine = (unsigned)dt < (unsigned)C::WTM && !(dt & 4);
      if (__builtin_amdgcn_ballot_w64(mine)) {
        int dsel = dt;
        asm volatile("" : "+v"(dsel));  // keeps the select inside the branch (not speculated)
        const float z = select_row<C>(acc, nb, dsel);
        if (mine) p.zt[tok] = z;
      }
      part += xor32(part);
      if (h == 0) red[wm][col] = part;
    }
    // Rows of this wave's block: tokens n0 + wn*WTN + (0..WTN-1), vocabulary vrow0 + (0..WTM-1).
    if constexpr (WITH_U) store_staged_tokmajor<C, BUF_NT, EDGE>(ub, p.ut, p.Npad, p.Vp, n0 + wn * C::WTN, vrow0, lane);
  };
  const bool inside = m0 + C::TM <= p.V && n0 + C::TN <= p.N;
  if (!SPLIT && p.ut) {
    if (inside) epilogue(std::true_type{}, std::false_type{});
    else epilogue(std::true_type{}, std::true_type{});
  } else {
    if (inside) epilogue(std::false_type{}, std::false_type{});
    else epilogue(std::false_type{}, std::true_type{});
  }
  __syncthreads();
  for (int t = threadIdx.x; t < C::TN; t += C::THREADS) {
    const int tok = n0 + t;
    if (tok >= p.N) continue;
    if constexpr (SPLIT && C::WTM == 128) {
#pragma unroll
      for (int w = 0; w < C::WM; ++w)
        if (m0 + w * C::WTM < p.V) p.partial[(size_t)(tm * C::WM + w) * p.N + tok] = red[w][t];
    } else {
      float s = 0.0f;
#pragma unroll
      for (int w = 0; w < C::WM; ++w) s += red[w][t];
      p.partial[(size_t)tm * p.N + tok] = s;
    }
  }
}

// Evaluation head (src/algebraic/evaluation.py:13-23 with the argmax of
// src/algebraic/benchmarking.py:178-188): z^T = E h^T as in the forward. The scorer's
// log_softmax(n asinh(z/c)) has no clamp, so the weights are evaluated relative to the largest
// logit z_m of a group of logits: w' = (rho(z/c) rho(-z_m/c))^n = exp(n (asinh(z/c) - asinh(z_m/c)))
// <= 1, which neither overflows however large the logits grow nor loses the group's leading
// terms. The epilogue keeps, per token and vocabulary tile, the tile's largest logit with its
// first index (the argmax), the sum of w' relative to that logit, and the target logit.
// Nothing per (token, vocab) pair is stored; head_eval_stats_kernel combines the tiles.

template <class C, int L2N>
__global__ __launch_bounds__(C::THREADS, head_waves_per_simd<C>()) void head_eval_kernel(HeadParams p) {
  __shared__ float red[C::WM][C::TN];
  __shared__ float redm[C::WM][C::TN];
  __shared__ int redi[C::WM][C::TN];
  const int nbm = (p.V + C::TM - 1) / C::TM, nbn = (p.N + C::TN - 1) / C::TN;
  int tm, tn;
  xcd_tile(blockIdx.x, nbm, nbn, tm, tn);
  const int m0 = tm * C::TM;  // vocab
  const int n0 = tn * C::TN;  // tokens
  GemmOperand A{p.E, p.d, p.V, p.d, (long)p.V * p.d}, B{p.h, p.d, p.N, p.d, (long)p.N * p.d};
  floatx16 acc[C::MB][C::NB];
  gemm_tile<KMAJOR, KMAJOR, C>(A, B, m0, n0, 0, p.d, acc);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int wm, wn;
  wave_coords<C>(wm, wn);
  const float inv_c = p.inv_c;
  const int vrow0 = m0 + wm * C::WTM;
  const bool inside = m0 + C::TM <= p.V;
#pragma unroll
  for (int nb = 0; nb < C::NB; ++nb) {
    const int col = wn * C::WTN + nb * 32 + l32;
    const int tok = n0 + col;
    const int tgt = tok < p.N ? p.targets[tok] : -1;
    // This lane's largest logit, its first index (the lane's vocabulary rows increase with
    // (mb, i)) and the sum of weights relative to it.
    float zm, part, sh;
    int im;
    bool done = false;
    if (inside) {
      // All rows live: the maximum alone, then the row that holds it, from the last to the first
      // (three instructions a logit where the ordered form below takes about ten: 148 -> 130 us at
      // N 1531, d 1024, V 32768).
      zm = acc[0][nb][0];
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) zm = fmaxf(zm, acc[mb][nb][i]);
      int row = 0;
#pragma unroll
      for (int mb = C::MB - 1; mb >= 0; --mb)
#pragma unroll
        for (int i = 15; i >= 0; --i) row = acc[mb][nb][i] == zm ? mb * 32 + 8 * (i >> 2) + (i & 3) : row;
      im = vrow0 + 4 * h + row;
      sh = eval_rho(-zm * inv_c);
      part = 0.0f;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) part += pow2n<L2N>(eval_rho(acc[mb][nb][i] * inv_c) * sh, p.log2n);
      done = part == part;  // a NaN or infinite logit makes the sum NaN
    }
    if (!done) {  // rows past V, and logits that are not finite: an order over each logit
      zm = -INFINITY;
      im = EVAL_NO_INDEX;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int v = vrow0 + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
          const float z = acc[mb][nb][i];
          // Rows increase along the lane: take z if it is larger, or the first NaN.
          if (v < p.V && !(z <= zm) && zm == zm) { zm = z; im = v; }
        }
      }
      sh = eval_rho(-zm * inv_c);
      part = 0.0f;
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int v = vrow0 + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
          if (v < p.V) part += pow2n<L2N>(eval_rho(acc[mb][nb][i] * inv_c) * sh, p.log2n);
        }
      }
    }
    // The target logit, as in the training forward.
    const int dt = tgt - vrow0 - 4 * h;
    const bool hit = (unsigned)dt < (unsigned)C::WTM && !(dt & 4);
    if (__builtin_amdgcn_ballot_w64(hit)) {
      int dsel = dt;
      asm volatile("" : "+v"(dsel));  // keeps the select inside the branch (not speculated)
      const float z = select_row<C>(acc, nb, dsel);
      if (hit && tgt < p.V) p.zt[tok] = z;
    }
    // The other lane half holds the same token's remaining rows of this wave's block.
    const float pz = __shfl_xor(zm, 32, 64);
    const float pp = __shfl_xor(part, 32, 64);
    const int pi = __shfl_xor(im, 32, 64);
    const bool take = pi != EVAL_NO_INDEX && eval_better(pz, pi, zm, im);
    const float zn = take ? pz : zm;
    const float mine = part == 0.0f ? 0.0f : part * eval_rescale<L2N>(zm, zn, inv_c, p.log2n);
    const float other = pp == 0.0f ? 0.0f : pp * eval_rescale<L2N>(pz, zn, inv_c, p.log2n);
    if (take) { zm = pz; im = pi; }
    if (h == 0) { red[wm][col] = mine + other; redm[wm][col] = zm; redi[wm][col] = im; }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < C::TN; t += C::THREADS) {
    const int tok = n0 + t;
    float m = -INFINITY;
    int ix = EVAL_NO_INDEX;
#pragma unroll
    for (int w = 0; w < C::WM; ++w)  // waves cover increasing vocabulary rows
      if (redi[w][t] != EVAL_NO_INDEX && eval_better(redm[w][t], redi[w][t], m, ix)) { m = redm[w][t]; ix = redi[w][t]; }
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < C::WM; ++w)
      if (red[w][t] != 0.0f) s += red[w][t] * eval_rescale<L2N>(redm[w][t], m, inv_c, p.log2n);
    if (tok < p.N) {
      p.partial[(size_t)tm * p.N + tok] = s;
      p.pmax[(size_t)tm * p.N + tok] = m;
      p.pidx[(size_t)tm * p.N + tok] = ix;
    }
  }
}

// The per-token reductions over vocabulary tiles below read one value per tile (stride N) and
// combine them in tile order within each wave's range of tiles; the loads are issued TB at a
// time so their latencies overlap, while the order of the combining steps stays that of a
// plain loop.
constexpr int TB = 16;

// log p(target) = log_softmax(n asinh(z/c))[t] (src/algebraic/evaluation.py:13-23) from the
// tiles' (largest logit, shifted sum) pairs: with z_m the largest logit of the row and
// L = sum over tiles of S_tile (rho(z_tile/c) rho(-z_m/c))^n = sum_v (rho(z_v/c) rho(-z_m/c))^n,
//   log p = n (log rho(z_t/c) + log rho(-z_m/c)) - log L,
// all in the log domain so that neither large logits nor improbable targets overflow or
// underflow. argmax: the first index of the largest logit over the tiles in vocabulary order
// (the first NaN if there is one, as jnp.argmax).
// 64 tokens per workgroup (lane = token, so each tile row is read as 256 contiguous bytes);
// the EVQ waves take consecutive ranges of the tiles, and their argmax candidates and partial
// sums are combined in range order through LDS. One token per thread over all the tiles left
// three quarters of the SIMDs idle at N = 16384: 48 us against 20.5 us with eight ranges in a
// kernel trace (HIP events: 27 us with four ranges, 24 us with eight).
constexpr int EVQ = 8;  // tile ranges (waves) per token
__global__ __launch_bounds__(64 * EVQ) void head_eval_stats_kernel(HeadParams p, int nvt) {
  __shared__ float sm[EVQ][64];
  __shared__ int si[EVQ][64];
  __shared__ float sl[EVQ][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int tok = blockIdx.x * 64 + lane;
  const bool live = tok < p.N;
  const int per = (nvt + EVQ - 1) / EVQ;
  const int t0 = min(nvt, q * per), t1 = min(nvt, t0 + per);
  float m = -INFINITY;
  int ix = EVAL_NO_INDEX;
  auto take = [&](float pm, int pi) {
    if (pi != EVAL_NO_INDEX && eval_better(pm, pi, m, ix)) { m = pm; ix = pi; }
  };
  if (live) {
    int t = t0;
    for (; t + TB <= t1; t += TB) {
      float vm[TB];
      int vi[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) {
        const size_t o = (size_t)(t + u) * p.N + tok;
        vm[u] = p.pmax[o];
        vi[u] = p.pidx[o];
      }
#pragma unroll
      for (int u = 0; u < TB; ++u) take(vm[u], vi[u]);
    }
    for (; t < t1; ++t) take(p.pmax[(size_t)t * p.N + tok], p.pidx[(size_t)t * p.N + tok]);
  }
  sm[q][lane] = m;
  si[q][lane] = ix;
  __syncthreads();
  m = -INFINITY;
  ix = EVAL_NO_INDEX;
#pragma unroll
  for (int r = 0; r < EVQ; ++r) take(sm[r][lane], si[r][lane]);
  // Sum of this range's tile sums, each moved onto m, in tile order.
  float l = 0.0f;
  auto add = [&](float s, float pm) {
    if (s != 0.0f) l += s * eval_rescale<0>(pm, m, p.inv_c, p.log2n);
  };
  if (live) {
    int t = t0;
    for (; t + TB <= t1; t += TB) {
      float vs[TB], vm[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) {
        const size_t o = (size_t)(t + u) * p.N + tok;
        vs[u] = p.partial[o];
        vm[u] = p.pmax[o];
      }
#pragma unroll
      for (int u = 0; u < TB; ++u) add(vs[u], vm[u]);
    }
    for (; t < t1; ++t) add(p.partial[(size_t)t * p.N + tok], p.pmax[(size_t)t * p.N + tok]);
  }
  sl[q][lane] = l;
  __syncthreads();
  if (q != 0 || !live) return;
  l = sl[0][lane];
#pragma unroll
  for (int r = 1; r < EVQ; ++r) l += sl[r][lane];
  // The target logit is written by the tile holding the target; out-of-range targets read 0.
  const int tgt = p.targets[tok];
  const float zt = tgt >= 0 && tgt < p.V ? p.zt[tok] : 0.0f;
  const float rel = zt == m ? 0.0f : logf(rho_exact(zt * p.inv_c)) + logf(rho_exact(-m * p.inv_c));
  p.logprob[tok] = (float)(1 << p.log2n) * rel - logf(l);
  // Both widths here: widening the indices afterwards was a launch of 7 us (N 1531).
  const int best = ix == EVAL_NO_INDEX ? 0 : ix;  // every logit -inf: index 0
  if (p.argmax) p.argmax[tok] = best;
  if (p.argmax64) p.argmax64[tok] = best;
}

// Per-token statistics and telemetry (fused_head.py:116-117, 219-229); with the residual
// schedule also l and the target entries of U.
// 64 tokens per workgroup, the vocabulary tiles split over EVQ waves as in the eval statistics:
// each wave sums its range in tile order, the ranges are added in range order.
__global__ __launch_bounds__(64 * EVQ) void head_stats_kernel(HeadParams p, int nvt) {
  __shared__ float sl[EVQ][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int tok = blockIdx.x * 64 + lane;
  const int per = (nvt + EVQ - 1) / EVQ;
  const int t0 = min(nvt, q * per), t1 = min(nvt, t0 + per);
  float part = 0.0f;
  if (tok < p.N) {
    int t = t0;
    for (; t + TB <= t1; t += TB) {
      float v[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) v[u] = p.partial[(size_t)(t + u) * p.N + tok];
#pragma unroll
      for (int u = 0; u < TB; ++u) part += v[u];
    }
    for (; t < t1; ++t) part += p.partial[(size_t)t * p.N + tok];
  }
  sl[q][lane] = part;
  __syncthreads();
  if (q != 0) return;
  float miss = 0.0f;
  if (tok < p.N) {
    float l = sl[0][lane];
#pragma unroll
    for (int r = 1; r < EVQ; ++r) l += sl[r][lane];
    const int n = 1 << p.log2n;
    const float st = inv_root(l, n);
    p.stat[tok] = st;
    // The forward wrote zt only where the target lies in [0, V); elsewhere it is 0
    // (fused_head.py:87 sums no column).
    const int tgt = p.targets[tok];
    const bool valid = tgt >= 0 && tgt < p.V;
    const float zt = valid ? p.zt[tok] : 0.0f;
    if (!valid) p.zt[tok] = 0.0f;
    const float x = fminf(zt / p.c, p.clamp);
    const float pt = ipow_rt(rho_exact(x) * st, n);
    p.pt[tok] = pt;
    miss = 1.0f - pt;
    if (p.lsum) p.lsum[tok] = l;
    if (p.ut) {
      if (valid) {
        float r;
        const float w = head_w(zt, p, r);
        p.ut[(size_t)tok * p.Vp + tgt] = f2bf((w - l) * r);
      }
    }
  }
  // This workgroup's sum of 1 - pt, by a fixed butterfly over the wave.
  for (int m = 32; m >= 1; m >>= 1) miss += __shfl_xor(miss, m, 64);
  if (lane == 0) p.obj_part[blockIdx.x] = miss;
}

__global__ __launch_bounds__(256) void head_obj_kernel(HeadParams p, int nblocks) {
  __shared__ float red[256];
  float s = 0.0f;
  for (int i = threadIdx.x; i < nblocks; i += 256) s += p.obj_part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.obj[0] = red[0] / (float)p.N;
}

// Recompute schedules: z^T again, dZ^T = s (p - y) r, token-major: rounded to bf16, or (SPLIT,
// f32 hidden states) as three bf16 planes whose sum is the f32 value times 2^split3_dz_exp(s). L2N > 0 fixes
// n = 2^L2N at compile time (0: taken from the parameters). Each wave's block is staged and
// written in whole token rows with 16-byte stores (default cache policy: the dh and dE products
// read dZ right after); edge tiles write the rows up to their end and the columns up to Vp too, of
// which nothing is read.
template <class C, int L2N, bool SPLIT>
__global__ __launch_bounds__(C::THREADS, head_waves_per_simd<C>()) void head_dz_kernel(HeadParams p) {
  if (SPLIT && *p.split_bad) return;
  const int nbm = (p.V + C::TM - 1) / C::TM, nbn = (p.N + C::TN - 1) / C::TN;
  int tm, tn;
  xcd_tile(blockIdx.x, nbm, nbn, tm, tn);
  const int m0 = tm * C::TM, n0 = tn * C::TN;
  const GemmOperand A = head_operand<SPLIT>(p.E, p.V, p.d, (long)p.V * p.d);
  const GemmOperand B = head_operand<SPLIT>(p.h, p.N, p.d, (long)p.N * p.d);
  floatx16 acc[C::MB][C::NB];
  bf16* ub = gemm_tile<KMAJOR, KMAJOR, C, SPLIT>(A, B, m0, n0, 0, p.d, acc);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int wm, wn;
  wave_coords<C>(wm, wn);
  float scale = head_grad_scale(p);
  if constexpr (SPLIT) scale = ldexpf(scale, split3_dz_exp(scale));
  const float inv_c = p.inv_c, clamp = p.clamp;
  const int vrow0 = m0 + wm * C::WTM;  // first vocab row of this wave
  __syncthreads();  // every wave is done reading the pipeline buffers
  auto epilogue = [&](auto edge) {
    constexpr bool EDGE = decltype(edge)::value;
#pragma unroll
    for (int nb = 0; nb < C::NB; ++nb) {
      const int tok = n0 + wn * C::WTN + nb * 32 + l32;
      const bool live = !EDGE || tok < p.N;
      const int dt = (live ? p.targets[tok] - p.v_off : -1) - vrow0 - 4 * h;  // target row relative to this lane's rows
      const float st = live ? p.stat[tok] : 0.0f;
      // The target entry, (t - 1) r s (y = 1), lies in this wave's rows for few tokens (WTM of V
      // rows), so it is formed behind a wave-uniform branch, as the forward selects the target
      // logit; every entry is formed with y = 0 and the target's replaced.
      const bool mine = (unsigned)dt < (unsigned)C::WTM && !(dt & 4);
      const bool some = __builtin_amdgcn_ballot_w64(mine);
      float utgt = 0.0f;
      int dsel = dt;
      if (some) {
        asm volatile("" : "+v"(dsel));  // keeps the select inside the branch (not speculated)
        const float x = fminf(select_row<C>(acc, nb, dsel) * inv_c, clamp);
        float r;
        const float t = pow2n<L2N>(rho_fast(x, r) * st, p.log2n);
        utgt = (t - 1.0f) * r * scale;
      }
#pragma unroll
      for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = fminf(acc[mb][nb][4 * g + e] * inv_c, clamp);
            float r;
            const float t = pow2n<L2N>(rho_fast(x, r) * st, p.log2n);
            u[e] = t * r * scale;  // (t - y) r s with y = 0; the target entry is patched below
          }
          u32x2 pk;
          pk[0] = pack_bf16x2(u[0], u[1]);
          pk[1] = pack_bf16x2(u[2], u[3]);
          *reinterpret_cast<u32x2*>(ub + ustage_at<C>(nb * 32 + l32, mb * 32 + 8 * g + 4 * h)) = pk;
        }
      }
      // The staged slot is overwritten (the same lane wrote it above; LDS keeps a wave's order).
      if (some && mine) ub[ustage_at<C>(nb * 32 + l32, dsel + 4 * h)] = f2bf(utgt);
    }
    store_staged_tokmajor<C, 0, EDGE>(ub, p.dzt, p.Npad, p.Vp, n0 + wn * C::WTN, vrow0, lane);
  };
  // SPLIT: blocks of 32 tokens x 64 vocabulary entries, whose three planes fit the wave's share
  // of the buffers together, so each value is formed once and split in registers.
  auto epilogue_split = [&]() {
    constexpr int SV = 64, SCH = SV / 8, PLANE = 32 * SV;
    static_assert(3 * PLANE <= gemm_share<KMAJOR, KMAJOR, C>() && C::WTM % SV == 0, "three planes fit the wave's share");
    auto at = [](int tl, int vl) { return tl * SV + (((vl >> 3) ^ (tl & (SCH - 1))) << 3) + (vl & 7); };
#pragma unroll
    for (int nb = 0; nb < C::NB; ++nb) {
      const int tok0 = n0 + wn * C::WTN + nb * 32, tok = tok0 + l32;
      const bool live = tok < p.N;
      const int dt = (live ? p.targets[tok] - p.v_off : -1) - vrow0 - 4 * h;
      const float st = live ? p.stat[tok] : 0.0f;
#pragma unroll
      for (int vb = 0; vb < C::WTM / SV; ++vb) {
#pragma unroll
        for (int m2 = 0; m2 < SV / 32; ++m2) {
          const int mb = vb * (SV / 32) + m2;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float u[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float x = fminf(acc[mb][nb][4 * g + e] * inv_c, clamp);
              float r;
              const float t = pow2n<L2N>(rho_fast(x, r) * st, p.log2n);
              u[e] = (t - (dt == mb * 32 + 8 * g + e ? 1.0f : 0.0f)) * r * scale;
            }
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) {
              u32x2 pk;
              pk[0] = pack_bf16x2(u[0], u[1]);
              pk[1] = pack_bf16x2(u[2], u[3]);
              *reinterpret_cast<u32x2*>(ub + pl * PLANE + at(l32, m2 * 32 + 8 * g + 4 * h)) = pk;
#pragma unroll
              for (int e = 0; e < 4; ++e)  // what this plane leaves: bf16 is the high half of an f32
                u[e] -= __builtin_bit_cast(float, e & 1 ? pk[e >> 1] & 0xffff0000u : pk[e >> 1] << 16);
            }
          }
          __builtin_amdgcn_sched_barrier(0);  // one 32 x 32 block's values at a time in registers
        }
        const int v0 = vrow0 + vb * SV, ch = lane % SCH;
        if (v0 + ch * 8 < p.Vp) {
#pragma unroll
          for (int pl = 0; pl < 3; ++pl) {
            bf16* out = p.dzt + ((size_t)pl * p.Npad + tok0) * p.Vp + v0 + ch * 8;
#pragma unroll
            for (int j = 0; j < 32 * SCH / 64; ++j) {
              const int tl = (64 / SCH) * j + lane / SCH;
              *reinterpret_cast<u32x4*>(out + (size_t)tl * p.Vp) =
                  *reinterpret_cast<const u32x4*>(ub + pl * PLANE + at(tl, ch * 8));
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if constexpr (SPLIT) epilogue_split();
  else if (m0 + C::TM <= p.V && n0 + C::TN <= p.N) epilogue(std::false_type{});
  else epilogue(std::true_type{});
}

// Residual schedule: hs = bf16(s h / l) (the row scale of dE = U'^T (s h / l)).
__global__ __launch_bounds__(256) void head_hscale_kernel(HeadParams p) {
  const float s = head_grad_scale(p);
  const size_t total8 = (size_t)p.N * p.d / 8;
  for (size_t c = (size_t)blockIdx.x * 256 + threadIdx.x; c < total8; c += (size_t)gridDim.x * 256) {
    const int row = (int)((c * 8) / p.d);
    const float f = s / p.lsum[row];
    bf16x8 x = *reinterpret_cast<const bf16x8*>(p.h + c * 8);
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = f2bf((float)x[j] * f);
    *reinterpret_cast<bf16x8*>(p.hs + c * 8) = y;
  }
}

// Store of a wave's WTM x WTN accumulator block, scaled per row and rounded to bf16, into a
// row-major matrix (interior tiles). Stored straight from the accumulators, each store
// instruction would cover 64 bytes of two rows at 2 bytes a lane; instead the block is staged
// in `stage` (this wave's share of the idle pipeline buffers) as [row][col] rows of WTN
// elements, 16-byte chunks XOR-swizzled by the row, and written back with 16-byte stores
// that cover whole 128-byte row segments. f(r) is the scale of block row r.
template <class C, class RowScale>
__device__ __forceinline__ void store_block_bf16(const floatx16 (&acc)[C::MB][C::NB], bf16* stage, bf16* out,
                                                 long ld, RowScale f) {
  constexpr int CH = C::WTN / 8;  // 16-byte chunks per staged row
  static_assert(CH <= 64 && 64 % CH == 0 && (CH & (CH - 1)) == 0, "staged row width");
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  auto at = [](int r, int c) { return r * C::WTN + (((c >> 3) ^ (r & (CH - 1))) << 3) + (c & 7); };
#pragma unroll
  for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      const float fr = f(r);
#pragma unroll
      for (int nb = 0; nb < C::NB; ++nb) stage[at(r, nb * 32 + l32)] = f2bf(acc[mb][nb][i] * fr);
    }
  }
  constexpr int RPS = 64 / CH;  // rows per store instruction
  const int c = lane % CH;
#pragma unroll
  for (int j = 0; j < C::WTM / RPS; ++j) {
    const int r = RPS * j + lane / CH;
    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + at(r, c * 8));
    *reinterpret_cast<u32x4*>(out + (long)r * ld + c * 8) = v;
  }
}


// dh = (U' or dZ) E: A stored token-major [n][v] (k-contiguous), B = E stored [v][d]
// (n-contiguous). The residual schedule scales token rows by s/l. When the product has too
// few output tiles to fill the chip (small N*d, long V) the vocabulary is split into
// dh_split ranges: each workgroup writes its f32 partial and head_dh_reduce_kernel sums them
// in a fixed order before the scale and the rounding. ACC (the streamed schedule's later
// vocabulary chunks, p.dh_accum 1 or 2): the tile of the f32 accumulator p.dh_part is read
// whole after the main loop (all loads issued before the first add) and added to the product,
// which then goes back to the accumulator (dh_accum 1) or, rounded, to dh (dh_accum 2).
// SPLIT (f32 hidden states): dZ and E as three bf16 planes each, the f32 result or its
// vocabulary partials, scaled back by 2^-split3_dz_exp, in p.dh_part.
template <class C, bool ACC, bool SPLIT>
__global__ __launch_bounds__(C::THREADS, head_waves_per_simd<C>()) void head_dh_kernel(HeadParams p) {
  if (SPLIT && *p.split_bad) return;
  const int nbm = (p.N + C::TM - 1) / C::TM, nbn = (p.d + C::TN - 1) / C::TN;
  int tr, tn;
  xcd_tile_rowmajor(blockIdx.x, nbm * p.dh_split, nbn, tr, tn);  // U panels streamed once
  // Split-major: the workgroups an XCD runs together share one vocabulary range, so its E
  // rows are read by every token tile there from L2 (C2: dh 0.658 -> 0.639 ms).
  const int split = tr / nbm, tm = tr - split * nbm;
  const int m0 = tm * C::TM;  // tokens
  const int n0 = tn * C::TN;  // d
  const int kbeg = min(p.V, split * p.dh_kchunk), kend = min(p.V, kbeg + p.dh_kchunk);
  const bf16* a = p.ut ? p.ut : p.dzt;
  const long apad = (long)p.Npad * p.Vp;
  const GemmOperand A{a, p.Vp, p.N, p.V, apad, 0, SPLIT ? apad : 0};
  const GemmOperand B = head_operand<SPLIT>(p.E, p.V, p.d, (long)p.V * p.d);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int wm, wn;
  wave_coords<C>(wm, wn);
  float* part = p.dh_part ? p.dh_part + (size_t)split * p.N * p.d : nullptr;
  floatx16 acc[C::MB][C::NB];
  bf16* stage = gemm_tile<KMAJOR, MNMAJOR, C, SPLIT>(A, B, m0, n0, kbeg, kend, acc);
  if constexpr (ACC) {
    // One 32 x 32 block at a time: its 16 loads are issued together, then added, and (dh_accum
    // 1) stored back to the accumulator.
    const bool back = p.dh_accum == 1;
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::NB; ++nb) {
        const int r0 = m0 + wm * C::WTM + mb * 32 + 4 * h, col = n0 + wn * C::WTN + nb * 32 + l32;
        float* blk = part + (size_t)r0 * p.d + col;
        float pv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int dr = 8 * (i >> 2) + (i & 3);
          pv[i] = r0 + dr < p.N && col < p.d ? blk[dr * p.d] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int dr = 8 * (i >> 2) + (i & 3);
          acc[mb][nb][i] += pv[i];
          if (back && r0 + dr < p.N && col < p.d) blk[dr * p.d] = acc[mb][nb][i];
        }
      }
    if (back) return;
  }
  const float s = p.ut ? head_grad_scale(p) : 1.0f;
  const float unscale = SPLIT ? ldexpf(1.0f, -split3_dz_exp(head_grad_scale(p))) : 1.0f;
  const bool to_dh = !part || ACC;  // bf16 output (ACC here: the last chunk)
  if (to_dh && m0 + C::TM <= p.N && n0 + C::TN <= p.d) {
    // Interior tile, bf16 output: the row scales s/l once per row (the expression of
    // head_hscale_kernel), then the staged 16-byte stores.
    __shared__ float fsc[C::TM];
    for (int t = threadIdx.x; t < C::TM; t += C::THREADS) fsc[t] = p.ut ? s / p.lsum[m0 + t] : 1.0f;
    __syncthreads();  // fsc is written and every wave is done with the pipeline buffers
    const int r0 = wm * C::WTM;
    store_block_bf16<C>(acc, stage, p.dh + (size_t)(m0 + r0) * p.d + n0 + wn * C::WTN, p.d,
                     [&](int r) { return fsc[r0 + r]; });
    return;
  }
#pragma unroll
  for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int tok = m0 + wm * C::WTM + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      if (tok >= p.N) continue;
      const float f = p.ut ? s / p.lsum[tok] : 1.0f;
#pragma unroll
      for (int nb = 0; nb < C::NB; ++nb) {
        const int col = n0 + wn * C::WTN + nb * 32 + l32;
        if (col >= p.d) continue;
        const size_t o = (size_t)tok * p.d + col;
        if (to_dh) p.dh[o] = f2bf(acc[mb][nb][i] * f);
        else part[o] = SPLIT ? acc[mb][nb][i] * unscale : acc[mb][nb][i];
      }
    }
  }
}

// dh = bf16(f * sum_s partial_s) over the vocabulary splits, summed in split order.
__global__ __launch_bounds__(256) void head_dh_reduce_kernel(HeadParams p) {
  const float s = p.ut ? head_grad_scale(p) : 1.0f;
  const size_t plane = (size_t)p.N * p.d;
  const size_t total8 = plane / 8;
  for (size_t c = (size_t)blockIdx.x * 256 + threadIdx.x; c < total8; c += (size_t)gridDim.x * 256) {
    const int row = (int)((c * 8) / p.d);
    const float4* src = reinterpret_cast<const float4*>(p.dh_part + c * 8);
    float4 a = src[0], b = src[1];
    for (int k = 1; k < p.dh_split; ++k) {
      const float4* q = reinterpret_cast<const float4*>(p.dh_part + k * plane + c * 8);
      const float4 x = q[0], y = q[1];
      a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      b.x += y.x; b.y += y.y; b.z += y.z; b.w += y.w;
    }
    const float f = p.ut ? s / p.lsum[row] : 1.0f;
    bf16x8 out;
    out[0] = f2bf(a.x * f); out[1] = f2bf(a.y * f); out[2] = f2bf(a.z * f); out[3] = f2bf(a.w * f);
    out[4] = f2bf(b.x * f); out[5] = f2bf(b.y * f); out[6] = f2bf(b.z * f); out[7] = f2bf(b.w * f);
    *reinterpret_cast<bf16x8*>(p.dh + c * 8) = out;
  }
}

// dE = (U' or dZ)^T (hs or h): A = U' stored token-major [n][v] (m-contiguous), B stored
// [n][d] (n-contiguous). Workgroups below de_full compute whole tiles, row-major inside each
// XCD's share (U panels streamed once); the rest compute token range (id - de_full) % de_split
// of tile de_full + (id - de_full) / de_split into an f32 tile of de_part, which
// head_de_tail_kernel sums.
// SPLIT (f32 hidden states): dZ and h as three bf16 planes each, the products scaled back by
// 2^-split3_dz_exp.
template <class C, bool SPLIT>
__global__ __launch_bounds__(C::THREADS, head_waves_per_simd<C>()) void head_de_kernel(HeadParams p) {
  if (SPLIT && *p.split_bad) return;
  const int nbn = (p.d + C::TN - 1) / C::TN;
  const int bid = blockIdx.x;
  int lin, kbeg = 0, kend = p.N, unit = -1;
  if (bid < p.de_full) {
    lin = xcd_contiguous(bid, p.de_full);
  } else {
    unit = bid - p.de_full;
    lin = p.de_full + unit / p.de_split;
    kbeg = (unit % p.de_split) * p.de_kchunk;
    kend = min(p.N, kbeg + p.de_kchunk);
  }
  const int tm = lin / nbn, tn = lin - tm * nbn;
  const int m0 = tm * C::TM;  // vocab
  const int n0 = tn * C::TN;  // d
  const bf16* a = p.ut ? p.ut : p.dzt;
  const bf16* b = p.ut ? p.hs : p.h;
  const long apad = (long)p.Npad * p.Vp;
  const GemmOperand A{a, p.Vp, p.N, p.V, apad, 0, SPLIT ? apad : 0};
  const GemmOperand B = head_operand<SPLIT>(b, p.N, p.d, (long)p.N * p.d);
  floatx16 acc[C::MB][C::NB];
  bf16* stage = gemm_tile<MNMAJOR, MNMAJOR, C, SPLIT>(A, B, m0, n0, kbeg, kend, acc);
  if constexpr (SPLIT) {
    const float unscale = ldexpf(1.0f, -split3_dz_exp(head_grad_scale(p)));
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][nb][i] *= unscale;
  }
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int wm, wn;
  wave_coords<C>(wm, wn);
  if (unit >= 0) {  // one token range of a split tile: the whole f32 tile, row-major
    float* part = p.de_part + (size_t)unit * C::TM * C::TN;
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = wm * C::WTM + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) part[r * C::TN + wn * C::WTN + nb * 32 + l32] = acc[mb][nb][i];
      }
    return;
  }
  if (!p.dE_f32 && m0 + C::TM <= p.V && n0 + C::TN <= p.d) {  // interior tile, bf16 output
    __syncthreads();  // every wave is done with the pipeline buffers
    store_block_bf16<C>(acc, stage,
                     reinterpret_cast<bf16*>(p.dE) + (size_t)(m0 + wm * C::WTM) * p.d + n0 + wn * C::WTN, p.d,
                     [](int) { return 1.0f; });
    return;
  }
#pragma unroll
  for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int v = m0 + wm * C::WTM + mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      if (v >= p.V) continue;
#pragma unroll
      for (int nb = 0; nb < C::NB; ++nb) {
        const int col = n0 + wn * C::WTN + nb * 32 + l32;
        if (col >= p.d) continue;
        const size_t o = (size_t)v * p.d + col;
        if (p.dE_f32) reinterpret_cast<float*>(p.dE)[o] = acc[mb][nb][i];
        else reinterpret_cast<bf16*>(p.dE)[o] = f2bf(acc[mb][nb][i]);
      }
    }
  }
}

// dE of a split tile: the de_split token-range tiles summed in range order, 32 rows of the
// tile per workgroup (grid: split tiles x HT_M / 32).
__global__ __launch_bounds__(256) void head_de_tail_kernel(HeadParams p) {
  if (p.split_bad && *p.split_bad) return;  // dE came whole from the f32 kernel
  const int nbn = (p.d + HT_N - 1) / HT_N;
  const int lin = p.de_full + blockIdx.x;
  const int tm = lin / nbn, tn = lin - tm * nbn;
  const float* part = p.de_part + (size_t)blockIdx.x * p.de_split * HT_M * HT_N;
#pragma unroll
  for (int c = 0; c < 32 * HT_N / 8 / 256; ++c) {
    const int e = (threadIdx.x + 256 * c) * 8;
    const int r = blockIdx.y * 32 + e / HT_N, col = e % HT_N;
    const int v = tm * HT_M + r, j0 = tn * HT_N + col;
    if (v >= p.V || j0 >= p.d) continue;
    const size_t o = (size_t)r * HT_N + col;
    float4 a = *reinterpret_cast<const float4*>(part + o), b = *reinterpret_cast<const float4*>(part + o + 4);
    for (int k = 1; k < p.de_split; ++k) {
      const float* q = part + (size_t)k * HT_M * HT_N + o;
      const float4 x = *reinterpret_cast<const float4*>(q), y = *reinterpret_cast<const float4*>(q + 4);
      a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      b.x += y.x; b.y += y.y; b.z += y.z; b.w += y.w;
    }
    const float vals[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const size_t out = (size_t)v * p.d + j0;  // d % 8 == 0: the 8 columns are in the row
    if (p.dE_f32) {
      float* dst = reinterpret_cast<float*>(p.dE) + out;
      *reinterpret_cast<float4*>(dst) = a;
      *reinterpret_cast<float4*>(dst + 4) = b;
    } else {
      bf16x8 o8;
#pragma unroll
      for (int t = 0; t < 8; ++t) o8[t] = f2bf(vals[t]);
      *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(p.dE) + out) = o8;
    }
  }
}

int head_token_pad(int N) { return ((N + HT_N - 1) / HT_N) * HT_N; }
int head_vocab_pitch(int V) { return (V + 7) / 8 * 8; }
int head_stat_blocks(int N) { return (N + 63) / 64; }

static int head_tiles(int tile, int M, int N) { return ((M + tile - 1) / tile) * ((N + tile - 1) / tile); }

// Tile side of the logit products (forward, dZ, evaluation): 128 where its tiles still run in one
// round. Then 256 x 256 tiles leave half the CUs idle or multiply padding (us, 256 / 128; N 128,
// d 1024, V 32768: forward 37 / 23, evaluation 46 / 24; N 512, d 512, V 8192: 22 / 15, 29 / 17);
// past one round the 128 tiles' epilogues, with nothing beside them on a CU, cost more than that
// (N 200, d 2048, V 32000: 59 / 74, 65 / 84; N 1000, d 1024, V 32768: 79 / 134, 93 / 163).
int head_logit_tile(int N, int V) { return head_tiles(128, V, N) <= 256 ? 128 : 256; }

// Vocabulary splits of the dh product on 256 x 256 tiles, for products with fewer than two rounds
// of tiles: minimise the rounds of 256 workgroups, ceil(tiles*S/256)/S of the whole product's k at
// 23.4 ns each, plus the f32 partials written and read at about 4.5 TB/s, keeping at least 512
// vocabulary entries per split; ties keep the smaller split count. (N 8192, d 768, V 50257, product
// and summing launch, us: S = 2 731 + 13, 4 777 + 21, 5 654 + 25, 8 657 + 37, 16 719 + 90.)
static int head_dh_split(int N, int d, int V) {
  const int tiles = head_tiles(HT_M, N, d);
  if (tiles >= 512) return 1;
  auto cost = [&](int s) {
    return std::ceil(tiles * (double)s / 256.0) / s * V * 0.0234 + (s > 1 ? 8e-6 / 4.5 * s * N * d : 0.0);
  };
  int best = 1;
  double best_cost = cost(1);
  for (int s = 2; s <= 16 && V / s >= 512; ++s)
    if (const double c = cost(s); c < best_cost - 1e-9) { best = s; best_cost = c; }
  return best;
}

// The dh product: that split, or, for few tokens, 128 x 128 tiles with up to 32 vocabulary splits,
// whichever takes less time. The time of a split is gemm_tile_time's form (rounds of 256 workgroups,
// a constant and a rate per k each), with constants of its own: f32 partials stored an element a
// lane, E read in rows of d, then the partials written and read and the summing launch. Fitted
// with it to 777 products: 0.3 % over the best form on average. A range of 128 tiles keeps 384 k at
// least. us, 256 / 128, with the summing launch (N, d, V): 128 1024 32768 77 / 44; 512 512 8192
// 46 / 32; 512 1024 50257 117 / 105; 700 1536 8192 56 / 77; 2500 1536 8192 87 / 125.
HeadDhPlan head_dh_plan(int N, int d, int V, int passes) {
  auto time = [&](int tile, int s) {
    const bool ragged = N % tile || d % tile;
    const int units = head_tiles(tile, N, d) * s, full = units / 256, rest = units % 256, rounds = full + (rest > 0);
    const double K = (double)head_dh_kchunk(V, s) * passes;
    const double t = tile == 256 ? 2.3 + rounds * 14.0 +
                                       K * (full * 0.025 + (rest > 0) * ((ragged ? 0.019 : 0.016) + 0.0076 * rest / 256.0))
                                 : 1.2 + rounds * (6.0 + K * (ragged ? 0.012 : 0.010));
    return t + (s > 1 ? 5.8 + 8e-6 * 0.087 * s * N * d : 0.0);
  };
  HeadDhPlan pl{256, head_dh_split(N, d, V), 0};
  double best = time(256, pl.split);
  if (head_tiles(256, N, d) < 256)
    for (int s = 1; s <= 32 && (s == 1 || V / s >= (passes == 1 ? 384 : 256)); s *= 2)
      if (const double t = time(128, s); t < best) {
        best = t;
        pl.tile = 128;
        pl.split = s;
      }
  pl.kchunk = head_dh_kchunk(V, pl.split);
  return pl;
}
int head_dh_kchunk(int V, int split) { return ((V + split - 1) / split + 127) / 128 * 128; }

// dE tiles past the last complete round of 256 workgroups are split over the tokens when that
// shortens the last round: S ranges per tile finish it in ceil(tail*S/256)/S of a tile's time
// instead of one (C2's 591 tiles: two full rounds, then 79 tiles x 3 ranges in a third of a
// tile's time). A range keeps at least 1024 tokens, and a split must save a quarter of a round
// (its f32 tiles are written and summed by head_de_tail_kernel); ties keep the smaller split.
// Products that do not fill a round take 128 x 128 tiles, unsplit, when gemm_tile_time says so; 6 us
// more for 256 tiles that reach past the matrix, which store an element a lane (N d V, us, 256 /
// 128: 100 896 8192 21.4 / 15.0; 128 1920 4096 19.6 / 12.8; 200 256 50257 22.7 / 35.1).
HeadDePlan head_de_plan(int N, int d, int V, int passes) {
  HeadDePlan pl;
  pl.tile = 256;
  pl.tiles = head_tiles(256, V, d);
  pl.full = pl.tiles;
  pl.split = 1;
  pl.kchunk = 0;
  const int full = pl.tiles / 256 * 256, tail = pl.tiles - full;
  if (tail == 0) return pl;
  int best = 1;
  double best_cost = 1.0;
  for (int s = 2; s <= 8 && N / s >= 1024; ++s) {
    const double cost = std::ceil(tail * (double)s / 256.0) / s;
    if (cost < best_cost - 1e-9) { best = s; best_cost = cost; }
  }
  if (best > 1 && best_cost <= 0.75) {
    pl.full = full;
    pl.split = best;
    pl.kchunk = ((N + best - 1) / best + 127) / 128 * 128;
    return pl;
  }
  const double K = (double)N * passes;
  const int tiles128 = head_tiles(128, V, d);
  if (full == 0 && gemm_tile_time(128, tiles128, K, V, d) <
                       gemm_tile_time(256, pl.tiles, K, V, d) + (V % 256 || d % 256 ? 6.0 : 0.0)) {
    pl.tile = 128;
    pl.tiles = pl.full = tiles128;
  }
  return pl;
}

template <class C, bool SPLIT>
static void launch_fwd_cfg(const HeadParams& p, hipStream_t st) {
  const dim3 grid(head_tiles(C::TM, p.V, p.N)), nt(C::THREADS);
  KTimer t(SPLIT ? "head_fwd_split" : "head_fwd", st);
  if (p.log2n == 3) hipLaunchKernelGGL((head_fwd_kernel<C, 3, SPLIT>), grid, nt, 0, st, p);
  else hipLaunchKernelGGL((head_fwd_kernel<C, 0, SPLIT>), grid, nt, 0, st, p);
}

hipError_t launch_head_fwd(const HeadParams& p, hipStream_t st) {
  const int tile = head_logit_tile(p.N, p.V);
  if (tile == 128) launch_fwd_cfg<HC128, false>(p, st);
  else launch_fwd_cfg<HC, false>(p, st);
  return launch_head_stats(p, (p.V + tile - 1) / tile, st);
}

// Statistics, telemetry and objective from the forward's per-tile partial sums (any tiling:
// vocab_tiles partial rows of N).
hipError_t launch_head_stats(const HeadParams& p, int vocab_tiles, hipStream_t st) {
  const int nb = head_stat_blocks(p.N);
  { KTimer t("head_stats", st); hipLaunchKernelGGL(head_stats_kernel, dim3(nb), dim3(64 * EVQ), 0, st, p, vocab_tiles); }
  { KTimer t("head_obj", st); hipLaunchKernelGGL(head_obj_kernel, dim3(1), dim3(256), 0, st, p, nb); }
  return hipGetLastError();
}

hipError_t launch_head_eval_stats(const HeadParams& p, int vocab_tiles, hipStream_t st) {
  KTimer t("head_eval_stats", st);
  hipLaunchKernelGGL(head_eval_stats_kernel, dim3(head_stat_blocks(p.N)), dim3(64 * EVQ), 0, st, p, vocab_tiles);
  return hipGetLastError();
}

template <class C>
static void launch_eval_cfg(const HeadParams& p, hipStream_t st) {
  const dim3 grid(head_tiles(C::TM, p.V, p.N)), nt(C::THREADS);
  KTimer t("head_eval", st);
  if (p.log2n == 3) hipLaunchKernelGGL((head_eval_kernel<C, 3>), grid, nt, 0, st, p);
  else hipLaunchKernelGGL((head_eval_kernel<C, 0>), grid, nt, 0, st, p);
}

hipError_t launch_head_eval(const HeadParams& p, hipStream_t st) {
  const int tile = head_logit_tile(p.N, p.V);
  if (tile == 128) launch_eval_cfg<HC128>(p, st);
  else launch_eval_cfg<HC>(p, st);
  return launch_head_eval_stats(p, (p.V + tile - 1) / tile, st);
}

// dh = (U' or dZ) E, and the sum over vocabulary splits when the product is split.
static void launch_head_dh(const HeadParams& p, hipStream_t st) {
  {
    KTimer t("head_dh", st);
    const dim3 grid(head_tiles(p.dh_tile, p.N, p.d) * p.dh_split);
    if (p.dh_accum) hipLaunchKernelGGL((head_dh_kernel<HC, true, false>), grid, dim3(HC::THREADS), 0, st, p);
    else if (p.dh_tile == 128) hipLaunchKernelGGL((head_dh_kernel<HC128, false, false>), grid, dim3(HC128::THREADS), 0, st, p);
    else hipLaunchKernelGGL((head_dh_kernel<HC, false, false>), grid, dim3(HC::THREADS), 0, st, p);
  }
  if (p.dh_split > 1) {
    const size_t chunks = (size_t)p.N * p.d / 8;
    const int blocks = (int)std::min<size_t>((chunks + 255) / 256, 4096);
    KTimer t("head_dh_reduce", st);
    hipLaunchKernelGGL(head_dh_reduce_kernel, dim3(blocks), dim3(256), 0, st, p);
  }
}

// dE = (U' or dZ)^T (hs or h), with the token split of head_de_plan when p carries one.
template <bool SPLIT>
static void launch_head_de(const HeadParams& p, hipStream_t st) {
  HeadParams q = p;
  const int tiles = head_tiles(p.de_tile, p.V, p.d);
  const bool split = p.de_split > 1 && p.de_part;
  if (!split) {
    q.de_full = tiles;
    q.de_split = 1;
  }
  const int tail = tiles - q.de_full;
  {
    KTimer t("head_de", st);
    const dim3 grid(q.de_full + tail * q.de_split);
    if (p.de_tile == 128) hipLaunchKernelGGL((head_de_kernel<HC128, SPLIT>), grid, dim3(HC128::THREADS), 0, st, q);
    else hipLaunchKernelGGL((head_de_kernel<HC, SPLIT>), grid, dim3(HC::THREADS), 0, st, q);
  }
  if (split) {
    KTimer t("head_de_tail", st);
    hipLaunchKernelGGL(head_de_tail_kernel, dim3(tail, HT_M / 32), dim3(256), 0, st, q);
  }
}

template <class C, bool SPLIT>
static void launch_dz_cfg(const HeadParams& p, hipStream_t st) {
  const dim3 grid(head_tiles(C::TM, p.V, p.N)), nt(C::THREADS);
  KTimer t(SPLIT ? "head_dz_split" : "head_dz", st);
  if (p.log2n == 3) hipLaunchKernelGGL((head_dz_kernel<C, 3, SPLIT>), grid, nt, 0, st, p);
  else hipLaunchKernelGGL((head_dz_kernel<C, 0, SPLIT>), grid, nt, 0, st, p);
}

static void launch_head_dz(const HeadParams& p, hipStream_t st) {
  if (head_logit_tile(p.N, p.V) == 128) launch_dz_cfg<HC128, false>(p, st);
  else launch_dz_cfg<HC, false>(p, st);
}

hipError_t launch_head_bwd(const HeadParams& p, hipStream_t st) {
  if (p.ut) {
    const size_t chunks = (size_t)p.N * p.d / 8;
    const int blocks = (int)std::min<size_t>((chunks + 255) / 256, 8192);
    { KTimer t("head_hscale", st); hipLaunchKernelGGL(head_hscale_kernel, dim3(blocks), dim3(256), 0, st, p); }
  } else {
    launch_head_dz(p, st);
  }
  launch_head_dh(p, st);
  launch_head_de<false>(p, st);
  return hipGetLastError();
}

// f32 hidden states on the bf16 matrix cores (p.E, p.h, p.dzt: three planes each; p.split_bad
// set): every launch returns at once when a value was out of the planes' range, and the f32
// kernels of head_f32.hip, launched after it, run instead.
//
// f32 values into three bf16 planes, each the bf16 nearest to what the planes before it leave;
// with 8 significant bits a plane the third leaves nothing. A value that is not zero and under
// SPLIT3_MIN (its last planes would be subnormal) or over SPLIT3_MAX, an infinity and a NaN set
// *bad. Bound by memory: 4 bytes read and 6 written an element.
__global__ __launch_bounds__(256) void head_split3_kernel(const float* src, bf16* dst, size_t n, int* bad) {
  bool off = false;
  for (size_t c = (size_t)blockIdx.x * 256 + threadIdx.x; c < n / 8; c += (size_t)gridDim.x * 256) {
    const float4 x = reinterpret_cast<const float4*>(src)[2 * c], y = reinterpret_cast<const float4*>(src)[2 * c + 1];
    float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = __builtin_fabsf(v[e]);
      off |= !((a >= SPLIT3_MIN && a <= SPLIT3_MAX) || a == 0.0f);
    }
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o[e] = f2bf(v[e]);
        v[e] -= (float)o[e];
      }
      *reinterpret_cast<bf16x8*>(dst + pl * n + 8 * c) = o;
    }
  }
  if (__builtin_amdgcn_ballot_w64(off) && (threadIdx.x & 63) == 0) *bad = 1;
}

// In the backward an upstream gradient that is not finite has no planes either.
__global__ void head_split_clear_kernel(HeadParams p, int* bad, bool backward) {
  *bad = backward && !(__builtin_fabsf(head_grad_scale(p)) < INFINITY);
}

// Planes of h and E, and *p.split_bad.
static void launch_head_split3(const HeadParams& p, bool backward, hipStream_t st) {
  KTimer t("head_split3", st);
  int* bad = const_cast<int*>(p.split_bad);
  hipLaunchKernelGGL(head_split_clear_kernel, dim3(1), dim3(1), 0, st, p, bad, backward);
  auto split = [&](const float* src, const bf16* dst, size_t n) {
    const int blocks = (int)std::min<size_t>((n / 8 + 255) / 256, 4096);
    hipLaunchKernelGGL(head_split3_kernel, dim3(blocks), dim3(256), 0, st, src, const_cast<bf16*>(dst), n, bad);
  };
  split(p.h32, p.h, (size_t)p.N * p.d);
  split(p.E32, p.E, (size_t)p.V * p.d);
}

void launch_head_fwd_split(const HeadParams& p, hipStream_t st) {
  launch_head_split3(p, false, st);
  if (head_logit_tile(p.N, p.V) == 128) launch_fwd_cfg<HC128, true>(p, st);
  else launch_fwd_cfg<HC, true>(p, st);
}

void launch_head_bwd_split(const HeadParams& p, hipStream_t st) {
  launch_head_split3(p, true, st);
  if (head_logit_tile(p.N, p.V) == 128) launch_dz_cfg<HC128, true>(p, st);
  else launch_dz_cfg<HC, true>(p, st);
  {
    HeadParams q = p;
    if (p.dh_split == 1) q.dh_part = p.dh32;
    KTimer t("head_dh_split", st);
    const dim3 grid(head_tiles(p.dh_tile, p.N, p.d) * p.dh_split);
    if (p.dh_tile == 128) hipLaunchKernelGGL((head_dh_kernel<HC128, false, true>), grid, dim3(HC128::THREADS), 0, st, q);
    else hipLaunchKernelGGL((head_dh_kernel<HC, false, true>), grid, dim3(HC::THREADS), 0, st, q);
  }
  launch_head_de<true>(p, st);
}

HeadParams head_vocab_chunk(const HeadParams& p, int v0, int vc) {
  HeadParams q = p;
  q.V = vc;
  q.Vp = head_vocab_pitch(vc);
  q.v_off = v0;
  const size_t rows = (size_t)v0 * p.d;
  if (p.E) q.E = p.E + rows;
  if (p.E32) q.E32 = p.E32 + rows;
  q.dE = p.dE_f32 ? static_cast<void*>(static_cast<float*>(p.dE) + rows) : static_cast<void*>(static_cast<bf16*>(p.dE) + rows);
  return q;
}

hipError_t launch_head_bwd_streamed(const HeadParams& p, int chunk, hipStream_t st) {
  const int nchunks = (p.V + chunk - 1) / chunk;
  for (int k = 0; k < nchunks; ++k) {
    HeadParams q = head_vocab_chunk(p, k * chunk, std::min(chunk, p.V - k * chunk));
    q.dh_tile = 256;
    q.dh_split = 1;
    q.dh_kchunk = head_dh_kchunk(q.V, 1);
    q.dh_part = nchunks > 1 ? p.dh_part : nullptr;
    q.dh_accum = k == 0 ? 0 : (k == nchunks - 1 ? 2 : 1);
    const HeadDePlan de = head_de_plan(p.N, p.d, q.V, 1);
    q.de_tile = de.tile;
    q.de_full = de.full;
    q.de_split = de.split;
    q.de_kchunk = de.kchunk;
    launch_head_dz(q, st);
    launch_head_dh(q, st);
    launch_head_de<false>(q, st);
  }
  return hipGetLastError();
}

}  // namespace alg
