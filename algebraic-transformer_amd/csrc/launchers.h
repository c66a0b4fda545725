// Host launchers of the gfx950 kernels (defined in the *.hip translation units).
#pragma once

#include <algorithm>
#include <cmath>

#include "attn_common.h"
#include "attn_prep.h"
#include "head_params.h"

namespace alg {

// The tile configurations of the bf16 products (gemm_core.h) are 256 x 256, 128 x 128 and, for the
// feed-forward, 64 x 64.
// Time in us of `units` workgroups of a tile configuration over k steps of K in all, fitted to
// the products of one short sequence and of the 1b block (M N K, measured us for tiles of 256 /
// 128 / 64, each in a captured graph with its launch):
//   1024  768 2048   39.3 / 20.8 / 11.0     768 4096 1024   25.4 / 14.7 / 19.6
//   1024  768 4096   69.5 / 37.2 / 19.2    2048  768 1024   23.2 / 12.6 /  8.3
//    512  512 2048   37.5 / 20.2 / 10.5    2048 2048 2048   41.8 / 25.1 / 36.7
// A 256 tile needs 14.8 ns per k alone on the chip and 23.4 ns when all CUs hold one (power); 128
// tiles 8 to 10 ns; 64 tiles 4 ns while a CU holds one, 8 ns for two. Small tiles move two or four
// times the operand bytes per multiplication, so they win only while the larger ones leave
// CUs idle.
inline double gemm_tile_time(int tile, int units, double K) {
  const double fill = std::min(1.0, units / 256.0), rounds = std::ceil(units / 256.0);
  if (tile == 256) return 9.0 + rounds * K * (0.0148 + 0.0086 * fill);
  if (tile == 128) return 4.4 + rounds * K * (0.008 + 0.002 * fill);
  return 2.8 + K * (units <= 512 ? 0.004 + 0.004 * std::max(0, units - 256) / 256.0 : std::ceil(units / 512.0) * 0.008);
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
hipError_t launch_ffn_gemm(const FfnGemmParams& g, int a_mode, int b_mode, hipStream_t st);
hipError_t launch_rms_norm_bwd(const RmsNormParams& p, float* dgain, hipStream_t st);

}  // namespace alg
