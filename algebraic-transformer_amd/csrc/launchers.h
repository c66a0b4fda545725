// Host launchers of the gfx950 kernels (defined in the *.hip translation units).
#pragma once

#include <algorithm>
#include <cmath>

#include "attn_common.h"
#include "attn_prep.h"
#include "head_params.h"

namespace alg {

// The tile configurations of the bf16 products (gemm_core.h) are 256 x 256, 128 x 128 and, for the
// feed-forward, 64 x 64. gemm_tile_time is the time in us of `units` workgroups of one of them over
// K, for an M x N result: rounds of 256 workgroups (512 of the 64 tiles, two to a CU), each a
// constant (the first copies and the epilogue, with nothing beside them) and a rate per k. The
// rates are lower while CUs stand idle (256 tiles: power; 64 tiles: one to a CU), and higher
// where tiles reach past the matrix, whose copies take a descriptor each. Fitted to 2876 products
// of the feed-forward (100 to 8000 tokens) and of the head (32 to 4096 tokens, V 1000 to 50257),
// each configuration timed on its own: the one chosen takes 1.0 % more than the best on average,
// and more than 1.04 times the 256 tiles in 13 of them (at most 1.26). Without the constant of each round and the ragged rates
// the same rule took up to 1.6 times the 256 tiles (M N K 1536 8448 197: 20.5 us, 32 on 792 tiles
// of 128). M N K, us for tiles of 256 / 128 / 64:
//   1024  768 2048   39.3 / 20.8 / 11.0     768 4096 1024   25.4 / 14.7 / 19.6
//   1024  768 4096   69.5 / 37.2 / 19.2    2048  768 1024   23.2 / 12.6 /  8.3
//   1024 8192  300   18.6 / 23.0 / 25.9    2048 1536 4224   42.8 / 39.5 / 58.4
inline double gemm_tile_time(int tile, int units, double K, int M, int N) {
  const bool ragged = M % tile || N % tile;
  if (tile == 256) {
    const int full = units / 256, rest = units % 256;
    return 1.4 + (full + (rest > 0)) * 9.0 +
           K * (full * 0.025 + (rest > 0) * ((ragged ? 0.017 : 0.014) + 0.0076 * rest / 256.0));
  }
  if (tile == 128) return 1.2 + std::ceil(units / 256.0) * (5.2 + K * (ragged ? 0.014 : 0.0088));
  const int full = units / 512, rest = units % 512;
  return 4.9 + (full + (rest > 0)) * 0.88 +
         K * ((full + (rest > 256)) * (ragged ? 0.0071 : 0.0068) + (rest > 0 && rest <= 256) * (ragged ? 0.0052 : 0.0042));
}

int attn_fwd_f32_query_block(int B, int H, int T);
hipError_t launch_attn_fwd(const AttnFwdParams& p, int D, bool bf16_io, int mode, hipStream_t st);
hipError_t launch_attn_bwd(const AttnBwdParams& p, int D, bool bf16_io, const int* modes, int nmodes,
                           hipStream_t st);
int attn_bwd_sink_blocks(int T);
int attn_prep_blocks(size_t rows);
hipError_t launch_attn_prep(const PrepParams& p, bool bf16_io, GuardParams g, hipStream_t st);
hipError_t launch_attn_guard(const GuardParams& g, hipStream_t st);
int attn_qk_prologue_blocks(int B, int H, int T, int D, bool bf16_io);
hipError_t launch_cayley_tables(const float* w, int half, int T, float* cos_out, float* sin_out, hipStream_t st);
hipError_t launch_attn_qk_prologue(const QkPrologueParams& p, bool bf16_io, GuardParams g, hipStream_t st);
hipError_t launch_attn_qk_prologue_bwd(const QkPrologueBwdParams& p, bool bf16_io, float* dq_gain, float* dk_gain,
                                       hipStream_t st);

int head_token_pad(int N);
int head_vocab_pitch(int V);
int head_stat_blocks(int N);
int head_logit_tile(int N, int V);
// `passes`: k passes of a product (1; 6 for f32 hidden states as three bf16 planes).
struct HeadDhPlan {
  int tile, split, kchunk;
};
HeadDhPlan head_dh_plan(int N, int d, int V, int passes);
int head_dh_kchunk(int V, int split);
struct HeadDePlan {
  int tile, tiles, full, split, kchunk;
};
HeadDePlan head_de_plan(int N, int d, int V, int passes);
hipError_t launch_head_fwd(const HeadParams& p, hipStream_t st);
hipError_t launch_head_bwd(const HeadParams& p, hipStream_t st);
// Rows [v0, v0 + vc) of the vocabulary as a head of its own: E, E32 and dE offset, V = vc,
// targets compared with v + v0.
HeadParams head_vocab_chunk(const HeadParams& p, int v0, int vc);
hipError_t launch_head_bwd_streamed(const HeadParams& p, int chunk, hipStream_t st);
hipError_t launch_head_eval(const HeadParams& p, hipStream_t st);
hipError_t launch_head_stats(const HeadParams& p, int vocab_tiles, hipStream_t st);
hipError_t launch_head_eval_stats(const HeadParams& p, int vocab_tiles, hipStream_t st);
int head_f32_vocab_tiles(int V);
bool head_f32_split(int N);
int head_f32_dh_split(int N, int d, int V);
int head_f32_dh_kchunk(int V, int split);
void launch_head_fwd_split(const HeadParams& p, hipStream_t st);
void launch_head_bwd_split(const HeadParams& p, hipStream_t st);
hipError_t launch_head_fwd_f32(const HeadParams& p, hipStream_t st);
hipError_t launch_head_bwd_f32(const HeadParams& p, hipStream_t st);
hipError_t launch_head_bwd_f32_streamed(const HeadParams& p, int chunk, hipStream_t st);
hipError_t launch_head_eval_f32(const HeadParams& p, hipStream_t st);
int rms_norm_max_d();
int rms_norm_blocks(int rows);
int rms_norm_gain_groups(int rows);
hipError_t launch_rms_norm_fwd(const RmsNormParams& p, hipStream_t st);
hipError_t launch_ffn_pack(const FfnPackParams& p, hipStream_t st);
hipError_t launch_ffn_fwd(const FfnParams& p, hipStream_t st);
hipError_t launch_ffn_dy(const FfnParams& p, hipStream_t st);
struct FfnGemmPlan {
  int tile, tiles, full, split, kchunk;
  size_t ws_bytes;  // f32 tiles of the split tiles
};
FfnGemmPlan ffn_gemm_plan(int M, int N, int K);
int ffn_gate_up_tile(int N, int F, int d);
int ffn_dy_tile(int N, int F, int dm);
hipError_t launch_ffn_gemm(const FfnGemmParams& g, int a_mode, int b_mode, hipStream_t st);
hipError_t launch_rms_norm_bwd(const RmsNormParams& p, float* dgain, hipStream_t st);

}  // namespace alg
