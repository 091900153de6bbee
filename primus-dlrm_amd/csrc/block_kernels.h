// Kernels of the OneTrans block that live in their own translation units, with
// the host-side launchers the block and stack entry points call.
#pragma once

#include "pdm_common.h"

namespace pdm {

// Q/K/V projection with RMSNorm1 in front:
//   Q[b, t - (kv - q_len)] (kept tail tokens), K[b, t], V^T[b, h, :, t] = bf16(bf16(RMSNorm1(x[b, t])) . Wqkv^T)
// S tokens (t < n_s) use the shared weight, NS token n_s + g uses the weight of token g.
struct QkvArgs {
  const float* x;         // fp32 rows, (b, t) at x + b * x_bstride + t * D
  int64_t x_bstride;      // elements between samples of x
  const float* norm_w;    // RMSNorm1 weight [D]
  const uint16_t* W;      // [3D, D] bf16 (S tokens)
  const uint16_t* W_ns;   // [n_ns, 3D, D] bf16, or null when n_ns == 0
  uint16_t* q;            // [B, q_len, D]
  uint16_t* k;            // [B, kv, D]
  uint16_t* vt;           // [B, D / 64, 64, kv_pad]
  int B, kv, q_len, n_ns, kv_pad;  // kv_pad: V^T row stride, a multiple of 64
  // filled by the launcher: S tokens per sample, row tiles per sample / per NS token, all tiles
  int n_s, tps, tpg;
  int64_t n_tiles;
};

// Weight-stationary launch for d_model 256 (each wave keeps one head's Q, K and V weight columns in
// registers); returns PDM_ERR_UNSUPPORTED for other widths.
int launch_qkv_stationary(const QkvArgs& a, int D, hipStream_t s);

// Row projection (row_proj.hip): out = epilogue(bf16(RMSNorm(x)) . W^T) for fp32 rows (b, t) of D columns.  S tokens
// (t < n_s) use W, NS token n_s + g uses W_ns[g].
enum { ROWPROJ_QKV = 0, ROWPROJ_GELU = 1 };
struct RowProjArgs {
  const float* x;        // row (b, t) at x + b * in_bstride + t * D
  int64_t in_bstride;
  const float* norm_w;   // RMSNorm weight [D]
  const uint16_t* W;     // [N, D]
  const uint16_t* W_ns;  // [n_ns, N, D], or null when n_ns == 0
  int B, n_s, n_ns, N;
  // ROWPROJ_GELU: out row (b, t) at out + b * out_bstride + t * N; the normalised bf16 rows are also left in h (the
  // layout of x) unless it is null
  uint16_t* h;
  uint16_t* out;
  int64_t out_bstride;
  // ROWPROJ_QKV (N = 3D): as QkvArgs
  uint16_t* q;
  uint16_t* k;
  uint16_t* vt;
  int kv, q_len, kv_pad;
  // filled by the launcher: tokens t < n_blk run in 32-token blocks of a sample, the n_tok behind them token by token
  int n_blk, n_tok, tiles_b, blocks_per_sample, wgs_s, wgs_tok, split_s, split_tok;
};
int launch_row_proj(const RowProjArgs& a, int D, int epi, hipStream_t s);

// Residual projection (resid_gemm.hip): out = A . W^T (rounded to bf16 with round_bf16) + res, fp32; S tokens (t < n_s) use W, NS token n_s + g
// uses W_ns[g].
struct ResidArgs {
  const uint16_t* A;     // bf16 row (b, t) at A + b * a_bstride + t * K
  int64_t a_bstride;
  const uint16_t* W;     // [N, K]
  const uint16_t* W_ns;  // [n_ns, N, K], or null when n_ns == 0
  int B, n_s, n_ns, N, K;  // N and K multiples of 128
  float* out;            // row (b, t) at out + b * out_bstride + t * N
  int64_t out_bstride;
  const float* res;      // row (b, t) at res + b * res_bstride + (t + res_toff) * N; may be out
  int64_t res_bstride;
  int res_toff;
  int round_bf16;
  // filled by the launcher
  int tiles_s, tiles_b;
};
int launch_resid_gemm(const ResidArgs& a, hipStream_t s);

}  // namespace pdm
