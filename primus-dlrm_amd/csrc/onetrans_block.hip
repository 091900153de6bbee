// OneTrans mixed-parameter block forward for gfx950 (bf16 MFMA).
//
// Semantics: OneTransBlock.forward(x, mask, q_len, n_s_tokens)
// (primus_dlrm/models/onetrans.py:207-231) under autocast(bf16)
// (primus_dlrm/training/dist_trainer.py:471) with an fp32 residual stream:
//   h1 = RMSNorm1(x)                         fp32 math, eps 1e-6     (:74-82)
//   qkv = h1 @ Wqkv^T  (shared for S-tokens, per-token for NS-tokens) (:124-139)
//   q  = q[:, kv - q_len:]                  pyramid tail              (:141-144)
//   o  = causal bottom-right softmax(q k^T / sqrt(dh)) v              (:62-67,148-161)
//   z  = o @ Wout^T + x[:, kv - q_len:]                               (:168-169,226-227)
//   y  = z + FFN(RMSNorm2(z)), FFN = W2 gelu_erf(W1 .), S shared / NS per token (:172-204)
// Every GEMM takes bf16 operands, accumulates in fp32 and rounds its output
// to bf16 (autocast), GELU runs in fp32 on the bf16 GEMM output and rounds
// to bf16, the residual additions run in fp32.  Exception: the FFN-down's
// output is added to z in fp32, not rounded to bf16 first (at most half a bf16
// ulp of the FFN output away from the autocast result).
//
// Launches per block: Q/K/V projection with RMSNorm1 in front (Q tail rows, K, and V transposed per head), attention,
// then either out-projection + FFN in one kernel or out-projection (+x tail -> z in y, resid_gemm.hip), FFN-up with
// RMSNorm2 in front (row_proj.hip), FFN-down (+z -> y, resid_gemm.hip).  Rows are (sample, token) pairs; S-token rows use
// the shared weight and NS-token rows the weight of their token, so one launch covers the shared GEMM and the 16
// per-token GEMMs.
//
// Attention design: one wave owns 32 queries of one (sample, head).  It
// computes S^T = K Q^T so that each lane holds one query's scores; the
// online softmax then needs a single cross-half exchange, and the fp32
// accumulator layout of S^T is already the B-operand layout of
// O^T = V^T P^T, so P never leaves registers.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "pdm_common.h"
#include "mfma_common.h"
#include "block_kernels.h"

namespace pdm {

struct GemmArgs {
  const uint16_t* A;  // bf16 rows: row (b, t) at A + b * a_bstride + t * K
  int64_t a_bstride;  // elements between samples
  const uint16_t* W;     // [N, K] shared (S-token) weight
  const uint16_t* W_ns;  // [n_ns, N, K] per-token weights, or null when shared by all rows
  int B;
  int n_s;    // tokens of the shared group per sample (tokens 0 .. n_s-1)
  int n_ns;   // per-token groups (tokens n_s .. n_s+n_ns-1); 0 when W_ns is null
  int N, K;
  int tiles_s, tiles_b;  // row tiles of the shared group, and per NS token
  int64_t total_blocks;
  // epilogue
  void* out;            // fp32 [B, T, D]
  int64_t out_bstride;  // elements between samples of out
  const float* res;     // residual fp32, row (b, t) at res + b * res_bstride + (t + res_toff) * K
  int64_t res_bstride;
  int res_toff;
  // the fused FFN
  const float* norm_w;    // RMSNorm2 weight
  const uint16_t* W2;     // FFN-down [D, F] shared
  const uint16_t* W2_ns;  // [n_ns, D, F]
  const uint16_t* Wo;     // FFN with the out-projection in front: Wout [D, D], shared by every token
};

// (sample, token) of row i of GEMM row tile mt, or b = -1 past the end.  Tiles
// 0 .. tiles_s-1 hold the shared group's rows (sample-major, token minor), the
// following tiles_b tiles per NS token hold that token's rows of every sample.
__device__ __forceinline__ void tile_row(const GemmArgs& a, int mt, int rows_per_tile, int i, int& b, int& t) {
  b = -1;
  t = 0;
  if (mt < a.tiles_s) {
    const int64_t r = (int64_t)mt * rows_per_tile + i;
    if (r < (int64_t)a.B * a.n_s) {
      b = (int)(r / a.n_s);
      t = (int)(r - (int64_t)b * a.n_s);
    }
  } else {
    const int g = (mt - a.tiles_s) / a.tiles_b;
    const int r = ((mt - a.tiles_s) - g * a.tiles_b) * rows_per_tile + i;
    if (r < a.B) {
      b = r;
      t = a.n_s + g;
    }
  }
}

// NS tiles in XCD-major order for a persistent grid of a multiple of 8 workgroups, which the dispatcher deals
// round-robin over the 8 XCDs (tile mt runs on XCD mt % 8): the NS tile that runs at position mt is the
// rank-th tile of the list sorted by (token % 8, token, tile), where rank is mt's place among the NS
// positions sorted by (mt % 8, mt).  When the counts agree (16 NS tokens, 8 tiles each), every tile of a
// token runs on one XCD, whose L2 then fetches the token's weights once instead of every XCD fetching every
// token's.  A bijection on the NS tiles for any sizes; S tiles are unchanged.
__device__ __forceinline__ int ns_tile_xcd_major(const GemmArgs& a, int mt) {
  if (mt < a.tiles_s) return mt;
  const int nt = a.n_ns * a.tiles_b;
  const int p = mt - a.tiles_s, cp = mt & 7;
  int rank = 0;
  for (int c = 0; c < cp; ++c) {
    const int q = (c - a.tiles_s) & 7;
    rank += q < nt ? (nt - 1 - q) / 8 + 1 : 0;
  }
  rank += (p - ((cp - a.tiles_s) & 7)) / 8;
  int pre = 0;
  for (int k = 0; k < 8; ++k) {
    const int ck = (k < a.n_ns ? (a.n_ns - 1 - k) / 8 + 1 : 0) * a.tiles_b;
    if (rank < pre + ck) {
      const int q = rank - pre;
      return a.tiles_s + (k + 8 * (q / a.tiles_b)) * a.tiles_b + q % a.tiles_b;
    }
    pre += ck;
  }
  return mt;  // not reached
}

// ---------------------------------------------------------------------------
// Out-projection and FFN in one kernel:  z = bf16(O . Wout^T) + x,  y = z + W2 . gelu(W1 . RMSNorm2(z))  for
// K = d_model = D, hidden F.
//
// Each of the NW waves owns 32 rows.  The out-projection runs in front: z^T = Wout . O^T accumulates straight into
// the y registers (lane l holds row l%32), every O fragment of the lane's row is requested up front and the Wout
// chunks (D rows x 64 columns, exactly one ring stage) go through the weight ring in front of the FFN chunks.  z is
// added to the residual x and normalised in registers; the RMSNorm2 values reach the B-operand layout of the FFN-up
// with one exchange of two words per 16-column step between the half-waves.  The FFN-down then accumulates on top of
// z, so y = z + FFN leaves the registers once and z never goes to memory.  The one difference from the reference's
// autocast rounding points: the FFN-down output is added to z in fp32 instead of being rounded to bf16 first, a
// difference of at most half a bf16 ulp of the FFN output.
//
// The hidden dimension is walked in chunks of 32 units: U^T = W1_c . h^T puts hidden units on the accumulator rows and
// token rows on the columns.  The FFN-up runs as 16x16x32 MFMAs into four independent accumulators (two 16-unit hidden
// blocks x two 16-token blocks): one exchange of the RMSNorm2 fragments per tile and one of the GELU values per chunk
// (v_permlane16_swap) keep both sides' operand reads single 16-byte LDS reads.  After GELU (fp32 on the bf16-rounded
// value, then bf16) those values are the B operand of y^T += W2[:, c] . G^T without leaving registers.
// W1 and W2 chunks go global -> LDS by LDS DMA into a 2-stage ring, chunk c + 1 issued right after the barrier that
// publishes chunk c.  Two workgroups of four waves share a CU (two waves per SIMD, 75 KB of LDS each): their barriers
// are independent, so one's GELU, prologue and epilogue run beside the other's MFMAs (one workgroup of eight waves
// keeps every wave of a SIMD in the same phase, and the hardware does not overlap them within a wave).
//
// The grid is persistent: WPS workgroups per CU walk the row tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...
// ---------------------------------------------------------------------------
template <int D, int NW, int WPS>
__global__ __launch_bounds__(NW * 64, WPS) void ffn_kernel(GemmArgs a) {
  constexpr int NST = 2;                     // ring stages
  constexpr int NT = NW * 64;                // threads
  constexpr int PF = NST - 1;                // chunks read ahead
  constexpr int KS = D / 16;
  constexpr int DB = D / 32;                 // 32-row blocks of the output (d)
  constexpr int TROWS = NW * 32;
  constexpr int W1_BYTES = 32 * 2 * D;       // 32 hidden units x D
  constexpr int W2_BYTES = D * 64;           // D outputs x 32 hidden units
  // one LDS block: the weight ring, reused by the epilogue's staging tile
  constexpr int RING_BYTES = NST * (W1_BYTES + W2_BYTES);
  __shared__ __attribute__((aligned(16))) char sRing[RING_BYTES];
  char (*sW1)[W1_BYTES] = reinterpret_cast<char (*)[W1_BYTES]>(sRing);
  char (*sW2)[W2_BYTES] = reinterpret_cast<char (*)[W2_BYTES]>(sRing + NST * W1_BYTES);
  __shared__ int s_rb[TROWS];
  __shared__ int s_rt[TROWS];
  __shared__ float sGelu[GELU_T_N];
  __shared__ __attribute__((aligned(16))) float sNw[D];  // RMSNorm2 weight

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  gelu_table_fill(sGelu, tid, NT);
  for (int i = tid; i < D; i += NT) sNw[i] = a.norm_w[i];
  const int F = a.N;
  const uint16_t* W1 = a.W;
  const uint16_t* W2 = a.W2;
  // the O fragments of a tile's rows, the out-projection's B operand: lane (fr, hf) holds row
  // wave * 32 + fr, columns 16 s + hf * 8 .. + 8 of 64-column chunk kc
  constexpr int DWO = D / 64;
  u32x4_t ofr[DWO][4];
  auto load_o = [&](int mt_, int fr_, int hf_) {
    int b, t;
    tile_row(a, mt_, TROWS, wave * 32 + fr_, b, t);
    // rows past the end read row 0, unused
    const uint16_t* orow = a.A + (b >= 0 ? (int64_t)b * a.a_bstride + (int64_t)t * D : 0) + hf_ * 8;
#pragma unroll
    for (int kc = 0; kc < DWO; ++kc)
#pragma unroll
      for (int s = 0; s < 4; ++s) ofr[kc][s] = *reinterpret_cast<const u32x4_t*>(orow + kc * 64 + s * 16);
  };

  // Weight chunk c goes from global memory straight into LDS (global_load_lds_dwordx4: lane l of a wave
  // writes the 16 bytes at the wave's LDS base + 16 l), so LDS piece o of a stage is loaded by thread
  // o mod NT, round o / NT, and the source address is what decides the layout.
  // W1 stage: row r = hidden unit c*32 + r, D columns in 2D bytes,
  // 16-byte piece v of the row at slot v ^ (r & 15), so the 32 rows of one fragment read hit distinct
  // bank groups.  W2 stage: W2[d, c*32 .. c*32+32) as D rows of 64 bytes, piece v at v ^ ((d >> 2) & 3).
  constexpr int L1 = W1_BYTES / 16 / NT;     // pieces per thread of a W1 chunk
  constexpr int L2 = W2_BYTES / 16 / NT;     // and of a W2 chunk
  static_assert(L1 * NT * 16 == W1_BYTES && L2 * NT * 16 == W2_BYTES, "chunk pieces must cover the threads");
  // Per-thread byte offsets of its pieces within chunk 0 (the chunk adds a uniform offset).  Piece p of a
  // thread is row p * RP + r0 of the stage (RP = NT / (D / 8) rows per round of pieces, r0 = tid / (D / 8)):
  // the multiple of 16 in that row index only moves the source by whole rows, so it goes into the scalar
  // base and the thread keeps one offset per distinct (p * RP) mod 16.  W2 pieces differ by whole groups of
  // NT / 4 rows (a scalar offset) and share one per-thread offset.
  constexpr int RP = NT / (D / 8);
  static_assert(RP * (D / 8) == NT && (RP >= 16 ? RP % 16 == 0 : 16 % RP == 0), "W1 piece rows");
  constexpr int NLO = RP >= 16 ? 1 : 16 / RP;  // distinct (p * RP) mod 16
  static_assert(NT % 64 == 0, "W2 pieces");
  uint32_t off1[NLO];
  {
    const int r0 = tid / (D / 8), slot = tid % (D / 8);
#pragma unroll
    for (int j = 0; j < NLO; ++j) {
      const int r = j * RP + r0;  // < 16
      off1[j] = (uint32_t)((r * D + ((slot ^ (r & 15)) << 3)) * 2);
    }
  }
  const uint32_t off2 = (uint32_t)(((tid >> 2) * F + (((tid & 3) ^ ((tid >> 4) & 3)) * 8)) * 2);
  // The DMA is issued from inline assembly: the compiler's own tracking of LDS DMA makes every later LDS
  // read wait for it.  Its completion is awaited explicitly (s_waitcnt vmcnt(0) before the barrier that
  // publishes a chunk and before the epilogue reuses the ring); the compiler's own vmcnt waits stay
  // correct with these loads outstanding, since vector memory loads complete in issue order.
  auto dma = [&](int c, int stg) {
    const uint64_t b1 = (uint64_t)(uintptr_t)W1 + (uint64_t)c * 32 * D * 2;
    const uint64_t b2 = (uint64_t)(uintptr_t)W2 + (uint64_t)c * 32 * 2;
#pragma unroll
    for (int p = 0; p < L1; ++p)
      lds_dma16(b1 + (uint64_t)(((p * RP) & ~15) * D * 2), off1[((p * RP) & 15) / (RP >= 16 ? 16 : RP)],
                (uint32_t)(uintptr_t)(sW1[stg] + (p * NT + wave * 64) * 16));
#pragma unroll
    for (int p = 0; p < L2; ++p)
      lds_dma16(b2 + (uint64_t)p * (NT / 4) * F * 2, off2, (uint32_t)(uintptr_t)(sW2[stg] + (p * NT + wave * 64) * 16));
  };
  const int nchunks = F / 32;
  constexpr unsigned kWaitDma = 0x0F70u | (unsigned)((PF - 1) * (L1 + L2));
  static_assert((PF - 1) * (L1 + L2) < 16, "vmcnt immediate");
  // Persistent: the workgroup walks the row tiles blockIdx.x, blockIdx.x + gridDim.x, ...
  for (int mt_run = blockIdx.x; mt_run < a.total_blocks; mt_run += gridDim.x) {
  const int mt = ns_tile_xcd_major(a, mt_run);
  // The lane's LDS and global offsets below derive from an opaque copy of the lane index taken per tile, so
  // the compiler recomputes them in each tile instead of holding them in registers through the prologue and
  // epilogue, where every register is taken.
  int lane;
  asm volatile("v_and_b32 %0, 63, %1" : "=v"(lane) : "v"(tid));
  const int fr = lane & 31, hf = lane >> 5;
  // every wave is done with the previous tile's staging tile (the ring) and row map
  __syncthreads();
  for (int i = tid; i < TROWS; i += NT) tile_row(a, mt, TROWS, i, s_rb[i], s_rt[i]);
  {
    const int64_t gsel = mt < a.tiles_s ? -1 : (mt - a.tiles_s) / a.tiles_b;
    W1 = gsel < 0 ? a.W : a.W_ns + gsel * (int64_t)F * D;
    W2 = gsel < 0 ? a.W2 : a.W2_ns + gsel * (int64_t)D * F;
  }
  __syncthreads();
  u32x4_t hfr[KS];
  f32x16_t y[DB];
  {
    constexpr int DW = D / 64;  // Wout chunks of 64 columns, each D rows x 128 bytes = one ring stage
    static_assert(DW % NST == 0, "FFN chunk c must keep stage c % NST");
    // Wout chunk kc: LDS row r (output feature) = Wout[r, kc*64 .. +64), rows 0 .. D/2 - 1 in the W1 part of
    // the stage, the rest in its W2 part; 16-byte piece v of a row at slot v ^ (r & 7)
    // piece p of a thread is row p * NT / 8 + tid / 8 (rows of 8 pieces, NT / 8 a multiple of 8): one
    // per-thread offset, the row group in the scalar base
    static_assert((NT / 8) % 8 == 0, "Wout pieces");
    const uint32_t offw = (uint32_t)(((tid >> 3) * D + (((tid & 7) ^ ((tid >> 3) & 7)) << 3)) * 2);
    auto dma_wo = [&](int kc, int stg) {
      const uint64_t b = (uint64_t)(uintptr_t)a.Wo + (uint64_t)kc * 128;
#pragma unroll
      for (int p = 0; p < L1; ++p)
        lds_dma16(b + (uint64_t)p * (NT / 8) * D * 2, offw, (uint32_t)(uintptr_t)(sW1[stg] + (p * NT + wave * 64) * 16));
#pragma unroll
      for (int p = L1; p < L1 + L2; ++p)
        lds_dma16(b + (uint64_t)p * (NT / 8) * D * 2, offw,
                  (uint32_t)(uintptr_t)(sW2[stg] + ((p - L1) * NT + wave * 64) * 16));
    };
    const int row = wave * 32 + fr;
    const int b = s_rb[row], t = s_rt[row];
    const bool valid = b >= 0;
    static_assert(DW == DWO, "Wout chunks");
    // every O fragment of the row (4 per Wout chunk) is requested up front, after the DMA of the first two
    // Wout chunks (both ring stages are free), so one memory latency covers the whole out-projection
    dma_wo(0, 0);
    dma_wo(1, 1);
    load_o(mt, fr, hf);
    const float* xrow = a.res + (valid ? (int64_t)b * a.res_bstride + (int64_t)(t + a.res_toff) * D : 0) + hf * 4;
    f32x4_t xv[DB][4];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) y[db][e] = 0.0f;
#pragma unroll
    for (int kc = 0; kc < DW; ++kc) {
      const int stg = kc % NST;
      // chunk kc's Wout rows have landed and every wave is done with the stage the next DMA fills.  Only DMA
      // pieces are counted (the compiler may issue the O loads later; it waits for those itself): at chunk 0
      // the L1 + L2 pieces of Wout chunk 1 may still be in flight, later chunks wait for everything.
      if (kc == 0) __builtin_amdgcn_s_waitcnt(0x0F70u | (unsigned)(L1 + L2));
      else __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
      __syncthreads();
      if (kc >= 1) {
        if (kc + 1 < DW) dma_wo(kc + 1, (kc + 1) % NST);
        else dma(0, (kc + 1) % NST);  // FFN chunk 0
      }
      if (kc == DW - 1) {
        // the residual of the first half of the outputs, before the last chunk's MFMAs
#pragma unroll
        for (int db = 0; db < DB / 2; ++db)
#pragma unroll
          for (int g = 0; g < 4; ++g) xv[db][g] = *reinterpret_cast<const f32x4_t*>(xrow + db * 32 + g * 8);
      }
      // z^T[db] += Wout[db rows, kc*64 + s*16 ..] . O^T: logical piece 2s + hf of row db*32 + fr
      u32x4_t wf[4 * DB];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const char* base = db < DB / 2 ? sW1[stg] + (db * 32 + fr) * 128 : sW2[stg] + ((db - DB / 2) * 32 + fr) * 128;
          wf[s * DB + db] = *reinterpret_cast<const u32x4_t*>(base + (((2 * s + hf) ^ (fr & 7)) << 4));
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int db = 0; db < DB; ++db) y[db] = mfma32x32x16(wf[s * DB + db], ofr[kc][s], y[db]);
      sched_mfma_ds_pipeline<4 * DB, 4>();
    }
    // z = bf16(O . Wout^T) + x[:, t + res_toff] in y (lane: row fr, outputs db*32 + g*8 + hf*4 + 0..3): the FFN
    // accumulates on top of it, so z never leaves the registers
    float ss = 0.0f;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      // the residual stays DB / 2 blocks ahead of its use
      if (db + DB / 2 < DB) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          xv[db + DB / 2][g] = *reinterpret_cast<const f32x4_t*>(xrow + (db + DB / 2) * 32 + g * 8);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float z = bf16_round(y[db][4 * g + j]) + xv[db][g][j];
          y[db][4 * g + j] = z;
          ss += z * z;
        }
      }
    }
    ss += __shfl_xor(ss, 32, 64);
    const float rms = 1.0f / sqrtf(ss / (float)D + 1e-6f);
    // RMSNorm2 -> the FFN-up B operand: 16-column step s (block db = s / 2, groups g0 = 2 (s % 2) and g0 + 1)
    // needs columns 16s + hf*8 + 0..7 in lane (fr, hf); the lane holds g0*8 + hf*4 + 0..3 and (g0+1)*8 + hf*4
    // + 0..3, so the half-waves swap one 4-column group
    const float* nw = sNw + hf * 4;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int db = s >> 1, g0 = 2 * (s & 1);
      const f32x4_t w0 = *reinterpret_cast<const f32x4_t*>(nw + db * 32 + g0 * 8);
      const f32x4_t w1 = *reinterpret_cast<const f32x4_t*>(nw + db * 32 + g0 * 8 + 8);
      const f32x16_t& zb = y[db];
      const int e0 = 4 * g0;
      const uint32_t a0 = pack_bf16x2((zb[e0] * rms) * w0.x, (zb[e0 + 1] * rms) * w0.y);
      const uint32_t a1 = pack_bf16x2((zb[e0 + 2] * rms) * w0.z, (zb[e0 + 3] * rms) * w0.w);
      const uint32_t b0 = pack_bf16x2((zb[e0 + 4] * rms) * w1.x, (zb[e0 + 5] * rms) * w1.y);
      const uint32_t b1 = pack_bf16x2((zb[e0 + 6] * rms) * w1.z, (zb[e0 + 7] * rms) * w1.w);
      const uint32_t r0 = (uint32_t)__shfl_xor((int)(hf ? a0 : b0), 32, 64);
      const uint32_t r1 = (uint32_t)__shfl_xor((int)(hf ? a1 : b1), 32, 64);
      hfr[s] = hf ? u32x4_t{r0, r1, b0, b1} : u32x4_t{a0, a1, r0, r1};
    }
  }

  // hfr (lane l: token l % 32, columns 16 s + 8 (l / 32) .. + 7 of step s) -> the B operand of the 16x16x32
  // FFN-up, two 16-token blocks tb: hfr[2 s2 + tb] of lane l then holds token 16 tb + l % 16, columns
  // 32 s2 + 16 (G & 1) + 8 (G >> 1) .. + 7 with G = l / 16.  Lanes l and l ^ 16 (same half-wave, tokens of the
  // two blocks) trade their pieces of odd and even steps: v_permlane16_swap exchanges the odd 16-lane rows
  // of its first operand with the even rows of its second.
#pragma unroll
  for (int s2 = 0; s2 < KS / 2; ++s2)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const auto sw = __builtin_amdgcn_permlane16_swap(hfr[2 * s2][w], hfr[2 * s2 + 1][w], false, false);
      hfr[2 * s2][w] = sw[0];
      hfr[2 * s2 + 1][w] = sw[1];
    }

  // The chunk loop is unrolled by the ring depth so that every stage index is a constant: the LDS reads of
  // stage k and the LDS DMA into stage (k + PF) % NST are then distinct objects to the compiler.
  for (int c0 = 0; c0 < nchunks; c0 += NST) {
#pragma unroll
    for (int k = 0; k < NST; ++k) {
      const int c = c0 + k;
      if (c >= nchunks) break;
      // chunks c .. c + PF - 1 are in LDS once every wave's DMA but the (PF - 1) (L1 + L2) pieces issued for
      // chunks c + 1 .. c + PF - 1 has landed (the wait; no other vector memory access is issued in the
      // loop, and they complete in issue order) and every wave has passed the barrier, which also means
      // every wave is done with chunk c - 1, whose stage receives chunk c + PF
      __builtin_amdgcn_s_waitcnt(kWaitDma);
      __syncthreads();
      // issued unconditionally (a branch around it costs the compiler its stage tracking): past the last chunk
      // it reloads the last chunk into the stage just freed, which no later chunk reads
      dma(min(c + PF, nchunks - 1), (k + PF) % NST);
      const char* w1 = sW1[k];
      uint32_t gp[8];
      // FFN-up with 16x16x32 MFMAs into four independent accumulators u4[hb][tb]: hidden units 16 hb + 4 G
      // + i (G = lane / 16, element i) of token 16 tb + lane % 16.  Step s2 takes the W1 fragment of row
      // 16 hb + lane % 16, piece 4 s2 + 2 (G & 1) + (G >> 1) (the columns the lane's hfr pieces hold).
      f32x4_t u4[2][2];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) u4[hb][tb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      // G = bf16(gelu(bf16(U))), half h2 = hidden block hb: lane l holds hidden units 16 h2 + 4 G + 0..3 of its
      // own token (block (l / 16) & 1) and of the token of lane l ^ 16; one exchange per word gives it hidden
      // units 16 h2 + 8 (l / 32) + 0..7 of token l % 32, the FFN-down's B operand for chunk c2 = h2
      auto gelu_half = [&](int h2) {
        float uv[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uv[i] = u4[h2][0][i];
          uv[4 + i] = u4[h2][1][i];
        }
        uint32_t t[4];
        gelu_lut_pack<8>(sGelu, uv, t);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const auto sw = __builtin_amdgcn_permlane16_swap(t[w], t[2 + w], false, false);
          gp[4 * h2 + w] = sw[0];
          gp[4 * h2 + 2 + w] = sw[1];
        }
      };
      {
        const int r16 = lane & 15, pofs = 2 * ((lane >> 4) & 1) + (lane >> 5);
        u32x4_t wf[KS];
#pragma unroll
        for (int s2 = 0; s2 < KS / 2; ++s2)
#pragma unroll
          for (int hb = 0; hb < 2; ++hb)
            wf[2 * s2 + hb] = *reinterpret_cast<const u32x4_t*>(w1 + (16 * hb + r16) * (2 * D) +
                                                                (((4 * s2 + pofs) ^ r16) << 4));
#pragma unroll
        for (int s2 = 0; s2 < KS / 2; ++s2)
#pragma unroll
          for (int hb = 0; hb < 2; ++hb)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) u4[hb][tb] = mfma16x16x32(wf[2 * s2 + hb], hfr[2 * s2 + tb], u4[hb][tb]);
        // 4 fragment reads ahead, then 4 MFMAs and the next step's 2 reads in turn
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < KS / 2 - 2; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
      }
      gelu_half(0);
      // The first half (G^T chunk c2 = 0) is computed before the FFN-down; the second half between the c2 = 0
      // MFMAs, which do not need it
      // FFN-down: y^T[db] += W2[db rows, chunk c] . G^T; chunk c2 of G^T holds hidden units
      // 16*c2 + hf*8 + 0..7, piece 2*c2 + hf of W2 row d, stored at (2*c2 + hf) ^ ((d >> 2) & 3)
      const char* w2 = sW2[k];
      {
        // (d >> 2) & 3 = (fr >> 2) & 3 for d = db*32 + fr
        u32x4_t wf[DB * 2];
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
          for (int db = 0; db < DB; ++db)
            wf[c2 * DB + db] =
                *reinterpret_cast<const u32x4_t*>(w2 + (db * 32 + fr) * 64 + (((2 * c2 + hf) ^ ((fr >> 2) & 3)) << 4));
        // the second GELU half has no dependence on the c2 = 0 MFMAs: the compiler's schedule interleaves them
        // (an explicit MFMA / DS / VALU group order kept more fragments live and spilled)
        gelu_half(1);
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
#pragma unroll
          for (int db = 0; db < DB; ++db) {
            const u32x4_t gb = {gp[4 * c2], gp[4 * c2 + 1], gp[4 * c2 + 2], gp[4 * c2 + 3]};
            y[db] = mfma32x32x16(wf[c2 * DB + db], gb, y[db]);
          }
        }
      }
    }
  }

  // Epilogue.  y[db][e] is output d = db*32 + (e/4)*8 + hf*4 + e%4 of row wave*32 + fr.
  // y already holds z + FFN (the FFN-down accumulated on top of z).  The values go through LDS (the weight ring is
  // free now) SEG outputs at a time, so that y is written as whole row segments of SEG outputs, with non-temporal
  // stores (y is streamed to memory; the next kernel reads it from there).
  constexpr int SEG = NW * 32 * (64 * 4 + 16) <= RING_BYTES ? 64 : 32;  // outputs per pass
  constexpr int SROW = SEG * 4 + 16;       // LDS row stride (bytes), padded against bank conflicts
  constexpr int NQ = D / SEG;              // passes
  constexpr int EK = 32 * (SEG / 4) / 64;  // 16-byte pieces per lane and pass
  static_assert(NW * 32 * SROW <= RING_BYTES, "epilogue staging must fit the weight ring");
  int64_t eoff[EK];  // piece k of this lane: its row's output offset + its 4 columns (pass 0), or -1
#pragma unroll
  for (int k = 0; k < EK; ++k) {
    const int piece = k * 64 + lane;     // 16-byte piece of the wave's 32 x SEG tile
    const int r = piece / (SEG / 4), c4 = piece - (piece / (SEG / 4)) * (SEG / 4);
    const int row = wave * 32 + r;
    const int b = s_rb[row];
    eoff[k] = b < 0 ? -1 : (int64_t)b * a.out_bstride + (int64_t)s_rt[row] * D + c4 * 4;
  }
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // the last DMA must land before the ring is reused
  __syncthreads();
  char* stage = sRing + wave * (32 * SROW);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
#pragma unroll
    for (int db2 = 0; db2 < SEG / 32; ++db2) {
      const int db = q * (SEG / 32) + db2;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4_t*>(stage + fr * SROW + (db2 * 32 + g * 8 + hf * 4) * 4) =
            f32x4_t{y[db][4 * g], y[db][4 * g + 1], y[db][4 * g + 2], y[db][4 * g + 3]};
    }
    // each wave reads back only its own tile; a wave's LDS accesses execute in order, so no barrier
#pragma unroll
    for (int k = 0; k < EK; ++k) {
      const int piece = k * 64 + lane;
      const int r = piece / (SEG / 4), c4 = piece - (piece / (SEG / 4)) * (SEG / 4);
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(stage + r * SROW + c4 * 16);
      if (eoff[k] >= 0)
        __builtin_nontemporal_store(v, reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(a.out) + eoff[k] + q * SEG));
    }
  }
  }  // row tiles
}

// ---------------------------------------------------------------------------
// Causal bottom-right attention, head dim 64.
// Q [B, q_len, H*64], K [B, kv, H*64], VT [B, H, 64, kv_pad] (bf16) -> O [B, q_len, H*64] bf16.
// Query i (0-based in the kept tail) sees keys j <= i + (kv - q_len).
// ---------------------------------------------------------------------------
struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* vt;
  uint16_t* o;
  int B, H, q_len, kv, kv_pad;  // kv_pad: keys held in LDS (kv rounded up to 32)
  int vt_ld;                     // V^T row stride in memory (kv rounded up to 64)
  float scale_log2;  // log2(e) / sqrt(64)
  int q_lds;         // attn_lds_kernel with 8 waves: Q of a head staged in LDS after K and V^T
  int parts;         // attn_lds_kernel with 8 waves: workgroups that share the query tiles of a head
};

// ---------------------------------------------------------------------------
// Persistent attention with the keys and values of a head resident in LDS.
// Each workgroup of NW waves walks the (sample, head) pairs blockIdx.x,
// blockIdx.x + gridDim.x, ...  K rows and V^T rows of a head are read from
// memory into registers while the previous head is computed, and written to
// LDS between two barriers, so the copy hides behind the attention math.
// With `parts` workgroups per head (one pass, the grid is parts * heads) workgroup
// part * heads + head takes every parts-th wave's tiles of its head; O goes over Q, and
// a wave uses only the Q rows of its own tiles, before it writes them.
// Each wave sweeps 32-query tiles over the key tiles up to its causal limit
// with no further barriers.  Query tiles go to waves in snake order of
// decreasing cost (the causal sweep of tile t covers t + 1 key tiles), so the
// waves of a head finish close together.  S^T = K Q^T puts a query per lane,
// online softmax in fp32, O^T += V^T P^T with P^T in registers.  Keys are
// stored in LDS with bits 2 and 3 of their index inside each group of 16
// swapped, so that the accumulator rows of S^T a lane holds for a 16-key step
// are 8 consecutive keys: the V^T operand is then one 16-byte read.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int swap23(int m) { return (m & ~12) | ((m & 4) << 1) | ((m & 8) >> 1); }

// Largest key count held in LDS (K 128 B + V^T 128 B per key).
constexpr int kAttnLdsMaxKeys = 608;

// One 32-query tile (queries 32 qt .. 32 qt + 31 of the kept tail) of causal bottom-right attention over
// one head's keys resident in LDS: K rows at sK (LDS row m holds key (m & ~15) | swap23(m & 15), 16-byte
// piece p at position p ^ ((m >> 1) & 7)) and V^T rows at sV (row d, piece pv of keys 8 pv .. at position
// pv ^ ((d >> 2) & 3)).  S^T = K Q^T per 32-key tile, online softmax in fp32, O^T += V^T P^T with P^T in
// registers; qf holds the tile's Q fragments; writes the tile's O rows (bf16) at o + qi * D.
// Softmax step of one 32-key tile: s holds the lane's 16 scores of its query (-inf where masked), m the
// running shift of the exponentials (log2 units, shared by the two lanes of a query), l the lane's share of
// the denominator, o the O^T accumulators.  The exponentials p = 2^(s * scale_log2 - m) go to pk as bf16
// pairs and their sum is returned; the normalised output does not depend on the shift.
//  LAZY = false: the tile's maximum first (the lane's 16 values; the other half-wave's only when m rises), m
//    raised when it exceeds m + 8, so every exponential is <= 2^8.
//  LAZY = true: the exponentials first; m is raised only when some lane's sum exceeds 2^16 or is not a
//    number (the first tile, where m = -inf), and then O and l are rescaled and the exponentials recomputed.
//    Every kept exponential is <= 2^16, and a tile with no new maximum costs no max reduction, at the cost
//    of the scores staying live until the check (about 14 more registers).
template <bool LAZY>
__device__ __forceinline__ float attn_tile_softmax(const f32x16_t& s, float scale_log2, float& m, float& l,
                                                   f32x16_t (&o)[2], uint32_t (&pk)[8]) {
  auto expo = [&]() {
    float ps = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale_log2, -m));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e + 1], scale_log2, -m));
      ps += p0 + p1;
      pk[e >> 1] = pack_bf16x2(p0, p1);
    }
    return ps;
  };
  auto lane_max = [&]() {  // the lane's 16 scores
    float mx = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
    for (int e = 3; e < 15; e += 2) mx = fmaxf(fmaxf(mx, s[e]), s[e + 1]);
    return fmaxf(mx, s[15]);
  };
  auto query_max = [](float mx) {  // with the other half of the wave (lane l ^ 32 holds the same query)
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
  };
  auto rescale = [&](float mt) {
    const float m_new = fmaxf(m, mt);
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);  // 0 on the first tile (m = -inf)
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 16; ++e) { o[0][e] *= alpha; o[1][e] *= alpha; }
  };
  // (scale_log2 > 0: the maximum of the scaled scores is the scaled maximum)
  if constexpr (LAZY) {
    const float ps = expo();
    if (!__builtin_amdgcn_ballot_w64(!(ps <= 0x1p16f))) return ps;
    rescale(query_max(lane_max()) * scale_log2);
    return expo();
  } else {
    // a query's maximum exceeds m + 8 exactly when one of its two lanes' does, so the exchange between the
    // half-waves is needed only when m rises
    const float mx = lane_max();
    if (__builtin_amdgcn_ballot_w64(mx * scale_log2 > m + 8.0f)) rescale(query_max(mx) * scale_log2);
    return expo();
  }
}

struct AttnTile {
  const char* sK;
  const char* sV;
  uint16_t* o;  // O row 0 of this (sample, head): o + qi * D for query qi
  int kvp, q_len, kv, D;
  float scale_log2;
};

template <bool LAZY>
__device__ __forceinline__ void attn_query_tile(const AttnTile& t, const int qt, const u32x4_t (&qf)[4], int fr,
                                                int hf) {
  const int qi0 = qt * 32;
  const int qi = qi0 + fr;
  const int off = t.kv - t.q_len;
  const int p_last = qi + off;  // last key this query sees
  const int q_last = min(qi0 + 31, t.q_len - 1);
  const int kv_end = min(t.kv, q_last + off + 1);

  f32x16_t o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) { o[0][e] = 0.0f; o[1][e] = 0.0f; }
  // m: the shift of the exponentials (log2 units), shared by the two lanes of a query; l: this lane's
  // share of the softmax denominator (attn_tile_softmax raises m only when the exponentials grow past 2^16).
  float m = -INFINITY, l = 0.0f;
  // key j0 + 16*(e/8) + hf*8 + e%8 of element e is visible iff 16*(e/8) + e%8 <= lim - j0
  const int lim = min(p_last, t.kv - 1) - hf * 8;
  const char* kp = t.sK + fr * 128;
  const char* vp0 = t.sV + fr * (2 * t.kvp);
  const char* vp1 = t.sV + (32 + fr) * (2 * t.kvp);
  int kofs[4], vofs[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) kofs[c] = ((2 * c + hf) ^ ((fr >> 1) & 7)) << 4;
#pragma unroll
  for (int c2 = 0; c2 < 2; ++c2) vofs[c2] = ((2 * c2 + hf) ^ ((fr >> 2) & 3)) << 4;  // (d >> 2) & 3, d = fr or 32 + fr

  // K and V^T fragments of a key tile are read one tile ahead of their MFMAs
  u32x4_t kf[4], vf[4];
  auto kread = [&](int j0, u32x4_t (&f)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = *reinterpret_cast<const u32x4_t*>(kp + j0 * 128 + kofs[c]);
  };
  // O^T[d][q] += V^T . P^T; chunk c2 of P^T holds keys j0 + 16*c2 + hf*8 + 0..7, which sit in
  // piece j0/8 + 2*c2 + hf of V^T row d, at position (j0/8) + ((2*c2 + hf) ^ ((d >> 2) & 3))
  auto vread = [&](int j0, u32x4_t (&f)[4]) {
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      f[2 * c2] = *reinterpret_cast<const u32x4_t*>(vp0 + j0 * 2 + vofs[c2]);
      f[2 * c2 + 1] = *reinterpret_cast<const u32x4_t*>(vp1 + j0 * 2 + vofs[c2]);
    }
  };
  kread(0, kf);
  vread(0, vf);
  for (int j0 = 0; j0 < kv_end; j0 += 32) {
    const int jn = j0 + 32 < kv_end ? j0 + 32 : j0;  // the last tile re-reads itself
    // S^T[key][q] = K . Q^T over the 32 LDS rows j0 .. j0+31 (row j0 + fr: piece p at p ^ ((fr >> 1) & 7))
    f32x16_t s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) s = mfma32x32x16(kf[c], qf[c], s);
    kread(jn, kf);
    // s[e] is LDS row j0 + (e/4)*8 + hf*4 + e%4, i.e. key j0 + 16*(e/8) + hf*8 + e%8
    if (j0 + 31 > qi0 + off || j0 + 32 > t.kv) {  // some key of the tile is masked for some query
      const int r = lim - j0;
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = (16 * (e >> 3) + (e & 7) <= r) ? s[e] : -INFINITY;
    }
    uint32_t pk[8];
    const float ps = attn_tile_softmax<LAZY>(s, t.scale_log2, m, l, o, pk);  // (rescales l and o first when m rises)
    l += ps;
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {
      const u32x4_t pb = {pk[4 * c2], pk[4 * c2 + 1], pk[4 * c2 + 2], pk[4 * c2 + 3]};
      o[0] = mfma32x32x16(vf[2 * c2], pb, o[0]);
      o[1] = mfma32x32x16(vf[2 * c2 + 1], pb, o[1]);
    }
    vread(jn, vf);
  }
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (qi < t.q_len) {
    // O may be written over Q: the calling wave has read every Q row of this tile, and no other wave reads them
    const float inv = 1.0f / l;
    uint16_t* orow = t.o + (int64_t)qi * t.D;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + g * 8 + hf * 4;
        u32x2_t w;
        w[0] = pack_bf16x2(o[db][4 * g] * inv, o[db][4 * g + 1] * inv);
        w[1] = pack_bf16x2(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv);
        *reinterpret_cast<u32x2_t*>(orow + d) = w;
      }
  }
}

// NP: 16-byte pieces per thread of K (and of V^T), kv_pad * 8 <= NP * 64 * NW.  NW = 8, one workgroup per
// CU; NW = 4 (two workgroups per CU, each on its own head) for heads of at most 4 query tiles, which would
// leave most of 8 waves idle.
template <int NP, int NW>
__global__ __launch_bounds__(NW * 64, 8 / NW) void attn_lds_kernel(AttnArgs a) {
  constexpr int NT = NW * 64;                // threads
  constexpr int RPR = NT / 8;                // K rows (and V^T rows) per copy round
  constexpr int VRS = 64 / RPR;              // rounds per set of the 64 V^T rows
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int kvp = a.kv_pad;                  // keys held (multiple of 32, <= kAttnLdsMaxKeys)
  char* sK = smem;                           // kvp rows x 128 bytes
  char* sV = smem + (int64_t)kvp * 128;      // 64 rows x 2*kvp bytes
  char* sQ = smem + (int64_t)kvp * 256;      // with q_lds: the head's Q rows, ntiles * 32 x 128 bytes
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int D = a.H * 64;
  const int BH = a.B * a.H;

  // Copy of one head, NP rounds of NT 16-byte pieces for K and for V^T:
  //  K: thread t holds LDS row m = RPR i + t / 8 (key (m & ~15) | swap23(m & 15)) and piece t % 8 of it,
  //     stored at piece position (t % 8) ^ ((m >> 1) & 7);
  //  V^T: thread t holds row d = t / 8 + RPR (i % VRS) and piece 8 (i / VRS) + t % 8 of it (keys
  //     64 (i / VRS) + 8 (t % 8) ..), stored at piece position (8 (i / VRS) + t % 8) ^ ((d >> 2) & 3).
  // Every per-round address is a fixed stride from round 0's (RPR is a multiple of 16).
  const int m0 = tid >> 3, p0 = tid & 7;
  const int key0 = (m0 & ~15) | swap23(m0 & 15);
  const int ppr = kvp >> 3;                  // pieces per V^T row
  char* const sk0 = sK + m0 * 128 + ((p0 ^ ((m0 >> 1) & 7)) << 4);
  char* const sv0 = sV + m0 * (2 * kvp) + ((p0 ^ ((m0 >> 2) & 3)) << 4);
  // Every read below is unconditional (out-of-range pieces read an in-range address and are zeroed
  // or skipped when stored), so that waits on the in-order memory counters never depend on a branch.
  u32x4_t kr[NP], vr[NP];
  auto gload = [&](int bh) {
    const int b = bh / a.H, h = bh - (bh / a.H) * a.H;
    const uint16_t* ksrc = a.k + (int64_t)b * a.kv * D + h * 64 + p0 * 8;
    const uint16_t* vsrc = a.vt + ((int64_t)bh * 64 + m0) * a.vt_ld;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      kr[i] = *reinterpret_cast<const u32x4_t*>(ksrc + (int64_t)min(RPR * i + key0, a.kv - 1) * D);
      vr[i] = *reinterpret_cast<const u32x4_t*>(vsrc + (int64_t)RPR * (i % VRS) * a.vt_ld + min(8 * (i / VRS) + p0, ppr - 1) * 8);
    }
  };
  auto sstore = [&]() {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (RPR * i + m0 < kvp)
        *reinterpret_cast<u32x4_t*>(sk0 + RPR * i * 128) = RPR * i + key0 < a.kv ? kr[i] : u32x4_t{0, 0, 0, 0};
      const int pv = 8 * (i / VRS) + p0;
      if (pv < ppr) {
        u32x4_t v = vr[i];
        if (pv * 8 + 8 > a.kv) {  // V^T beyond key kv - 1 is padding the QKV GEMM never wrote
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const int k0 = pv * 8 + 2 * w;
            if (k0 >= a.kv) v[w] = 0u;
            else if (k0 + 1 >= a.kv) v[w] &= 0xffffu;
          }
        }
        *reinterpret_cast<u32x4_t*>(sv0 + (int64_t)RPR * (i % VRS) * (2 * kvp) + 128 * (i / VRS)) = v;
      }
    }
  };

  const int ntiles = (a.q_len + 31) >> 5;
  const int parts = NW == 8 ? a.parts : 1;
  const int part = NW == 8 ? (int)blockIdx.x / BH : 0;  // 0 with one part: the grid is then at most BH
  // k-th tile of this wave in snake order (index into tiles sorted by decreasing cost), or -1
  auto tile_of = [&](int k) {
    const int nw = NW * parts, w = wave * parts + part;
    const int idx = nw * k + ((k & 1) ? nw - 1 - w : w);
    return idx < ntiles ? ntiles - 1 - idx : -1;
  };

  // Q fragments of query tile qt of (sample, head) pair p; rows past q_len read row q_len - 1 (their outputs
  // are never stored)
  auto qload = [&](int p, int qt, u32x4_t (&f)[4]) {
    const int b = p / a.H, h = p - (p / a.H) * a.H;
    const uint16_t* qbase = a.q + (int64_t)b * a.q_len * D + h * 64 + hf * 8;
    const int qi = min(qt * 32 + fr, a.q_len - 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = *reinterpret_cast<const u32x4_t*>(qbase + (int64_t)qi * D + c * 16);
  };
  // With q_lds, Q of head p goes to sQ by LDS DMA in 1 KB chunks of 8 rows: lane l of a chunk fills slot l
  // (row 8c + l / 8, position l % 8), which holds 16-byte piece (l % 8) ^ ((row >> 1) & 7) of the row, so
  // that a tile's fragment reads (32 rows, one piece each) spread over the banks; rows past q_len hold row
  // q_len - 1.  The wave's fragments of tile qt are then read from LDS.
  auto qdma = [&](int p) {
    const int b = p / a.H, h = p - (p / a.H) * a.H;
    const uint64_t qb = (uint64_t)(uintptr_t)(a.q + (int64_t)b * a.q_len * D + h * 64);
    const int r = lane >> 3, pos = lane & 7;
    for (int c = wave; c < ntiles * 4; c += NW) {
      const int row = 8 * c + r;
      const uint32_t off = (uint32_t)((min(row, a.q_len - 1) * D + ((pos ^ ((row >> 1) & 7)) << 3)) * 2);
      lds_dma16(qb, off, (uint32_t)(uintptr_t)(sQ + c * 1024));
    }
  };
  auto qread = [&](int qt, u32x4_t (&f)[4]) {
    const int row = qt * 32 + fr;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      f[c] = *reinterpret_cast<const u32x4_t*>(sQ + row * 128 + (((2 * c + hf) ^ ((row >> 1) & 7)) << 4));
  };
  // With 4 waves (heads of at most 4 query tiles: one tile per wave) the wave's tile of the next head has its
  // Q requested during this head, like the next head's K and V^T.
  constexpr bool kQNext = NW == 4;
  int bh = (int)blockIdx.x - part * BH;
  u32x4_t qf[4], qn[4];
  const bool q_lds = !kQNext && a.q_lds;
  if constexpr (kQNext) qload(bh, max(tile_of(0), 0), qf);
  if (q_lds) qdma(bh);
  gload(bh);
  for (;;) {
    __syncthreads();  // every wave is done with the previous head's LDS
    sstore();
    // Q of this head, requested before this head's copy, has landed (the copy's registers are consumed)
    if (q_lds) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
    const int b = bh / a.H, h = bh - (bh / a.H) * a.H;
    const int next = bh + (int)gridDim.x;
    const AttnTile at{sK, sV, a.o + (int64_t)b * a.q_len * D + h * 64, kvp, a.q_len, a.kv, D, a.scale_log2};
    auto process_tile = [&](const int qt, const u32x4_t (&qf)[4]) { attn_query_tile<(NP <= 8)>(at, qt, qf, fr, hf); };
    const int qt0 = tile_of(0), qt1 = tile_of(1);
    if constexpr (kQNext) {
      // this head's first tile was requested during the previous head; then the next head's copy and its
      // first tile's Q (O of a pair is written only by the workgroup that owns the pair, after its Q is read)
      __builtin_amdgcn_sched_barrier(0);
      gload(next < BH ? next : bh);
      if (next < BH) qload(next, max(qt0, 0), qn);
      __builtin_amdgcn_sched_barrier(0);
      if (qt0 >= 0) process_tile(qt0, qf);
      // further tiles (more than 4 per head): Q read at the start of the tile
      for (int kt = 1;; ++kt) {
        const int qt = tile_of(kt);
        if (qt < 0) break;
        qload(bh, qt, qf);
        process_tile(qt, qf);
      }
      if (next >= BH) break;
      qf[0] = qn[0];
      qf[1] = qn[1];
      qf[2] = qn[2];
      qf[3] = qn[3];
    } else {
      // A wave's first two tiles (all of them while q_len <= 512) have their Q requested before the next
      // head's copy, which then overlaps the whole head: memory reads complete in issue order for the
      // wait counter, so waiting for Q does not wait for the copy.  The code is straight-line up to the
      // second tile so that the compiler's waits count exactly; scheduling barriers keep the issue order.
      if (q_lds) {
        // every wave has at most two tiles: both read from LDS, then sQ is refilled with the next head's Q
        qread(max(qt0, 0), qf);
        qread(qt1 >= 0 ? qt1 : max(qt0, 0), qn);
        __syncthreads();
        if (next < BH) qdma(next);
        gload(next < BH ? next : bh);
      } else {
        qload(bh, max(qt0, 0), qf);
        qload(bh, qt1 >= 0 ? qt1 : max(qt0, 0), qn);
        __builtin_amdgcn_sched_barrier(0);
        gload(next < BH ? next : bh);  // in flight while this head is computed (the last head re-reads itself)
        __builtin_amdgcn_sched_barrier(0);
      }
      if (qt0 >= 0) process_tile(qt0, qf);
      if (qt1 >= 0) process_tile(qt1, qn);
      // tiles past the second (q_len > 512): Q read at the start of the tile
      for (int kt = 2;; ++kt) {
        const int qt = tile_of(kt);
        if (qt < 0) break;
        qload(bh, qt, qf);
        process_tile(qt, qf);
      }
      if (next >= BH) break;
    }
    bh = next;
  }
}

// ---------------------------------------------------------------------------
// Causal attention for heads whose keys do not fit in LDS (kv > kAttnLdsMaxKeys).  A workgroup of NW waves
// owns 32 NW consecutive queries of one (sample, head), one 32-query tile per wave, and streams the head's
// keys through LDS in chunks of 64: K rows and V^T rows in the layouts of attn_lds_kernel for 64 keys,
// double-buffered, the next chunk read into registers while the waves compute on the current one and written
// to the other buffer before the barrier that ends the chunk.  Each wave keeps its tile's online softmax
// state (shift m, denominator share l, O^T accumulators) in registers across the chunks and skips the chunks
// past its causal limit; the chunks stop at the workgroup's last visible key.  Workgroups take (sample, head,
// query block) items XCD-contiguously (the 8 XCDs take the workgroups in turn), so the query blocks of a head
// share one L2, and the longest query block of a head first.
// ---------------------------------------------------------------------------
constexpr int kStreamKeys = 64;  // keys per LDS chunk
#ifndef PDM_ATTN_STREAM_NW
#define PDM_ATTN_STREAM_NW 8  // waves (32-query tiles) per workgroup
#endif

template <int NW>
__global__ __launch_bounds__(NW * 64, 16 / NW) void attn_stream_kernel(AttnArgs a, int n_qb, int64_t n_items) {
  constexpr int NT = NW * 64;
  constexpr int PPT = kStreamKeys * 8 / NT;  // 16-byte pieces per thread of a chunk's K (and of its V^T)
  static_assert(PPT >= 1 && PPT * NT == kStreamKeys * 8, "chunk pieces must split evenly over the threads");
  __shared__ __attribute__((aligned(16))) char sbuf[2][2 * kStreamKeys * 128];  // per buffer: K 8 KB, V^T 8 KB
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int D = a.H * 64;
  // item = bh * n_qb + (n_qb - 1 - query block): XCD x takes the contiguous items x * q + min(x, r) ..
  int64_t item;
  {
    const int64_t id = blockIdx.x, q8 = n_items >> 3, r8 = n_items & 7, x = id & 7;
    item = x * q8 + (x < r8 ? x : r8) + (id >> 3);
  }
  const int bh = (int)(item / n_qb);
  const int qb = n_qb - 1 - (int)(item - (int64_t)bh * n_qb);
  const int b = bh / a.H, h = bh - (bh / a.H) * a.H;
  const int off = a.kv - a.q_len;
  const int wq0 = qb * (32 * NW);
  const int wq_last = min(wq0 + 32 * NW - 1, a.q_len - 1);
  const int kv_end = min(a.kv, wq_last + off + 1);  // keys the workgroup's queries see
  const int nchunks = (kv_end + kStreamKeys - 1) / kStreamKeys;
  const int qi0 = wq0 + wave * 32;
  const bool active = qi0 < a.q_len;  // wave-uniform
  const int qi = qi0 + fr;
  const int q_last = min(qi0 + 31, a.q_len - 1);
  const int w_end = active ? min(a.kv, q_last + off + 1) : 0;  // keys this wave's queries see
  const int p_last = qi + off;
  // key kb + j0 + 16*(e/8) + hf*8 + e%8 of element e is visible iff 16*(e/8) + e%8 <= lim - kb - j0
  const int lim = min(p_last, a.kv - 1) - hf * 8;

  // chunk copy: piece u = i * NT + tid; K: LDS row m = u / 8 (chunk key (m & ~15) | swap23(m & 15)), piece
  // u % 8 at position (u % 8) ^ ((m >> 1) & 7); V^T: row d = u / 8, piece pv = u % 8 (chunk keys 8 pv ..) at
  // position pv ^ ((d >> 2) & 3).  Reads are unconditional (clamped rows); keys past kv are stored as zeros.
  const uint16_t* kg = a.k + (int64_t)b * a.kv * D + h * 64;
  const uint16_t* vg = a.vt + (int64_t)bh * 64 * a.vt_ld;
  u32x4_t kr[PPT], vr[PPT];
  auto cload = [&](int cb) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      const int u = i * NT + tid, m = u >> 3, p = u & 7;
      const int key = cb + ((m & ~15) | swap23(m & 15));
      kr[i] = *reinterpret_cast<const u32x4_t*>(kg + (int64_t)min(key, a.kv - 1) * D + p * 8);
      vr[i] = *reinterpret_cast<const u32x4_t*>(vg + (int64_t)m * a.vt_ld + cb + p * 8);
    }
  };
  auto cstore = [&](int cb, int buf) {
    char* sK = sbuf[buf];
    char* sV = sbuf[buf] + kStreamKeys * 128;
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      const int u = i * NT + tid, m = u >> 3, p = u & 7;
      const int key = cb + ((m & ~15) | swap23(m & 15));
      *reinterpret_cast<u32x4_t*>(sK + m * 128 + ((p ^ ((m >> 1) & 7)) << 4)) =
          key < a.kv ? kr[i] : u32x4_t{0, 0, 0, 0};
      u32x4_t v = vr[i];
      if (cb + p * 8 + 8 > a.kv) {  // V^T beyond key kv - 1 is padding the Q/K/V projection never wrote
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int k0 = cb + p * 8 + 2 * w;
          if (k0 >= a.kv) v[w] = 0u;
          else if (k0 + 1 >= a.kv) v[w] &= 0xffffu;
        }
      }
      *reinterpret_cast<u32x4_t*>(sV + m * 128 + ((p ^ ((m >> 2) & 3)) << 4)) = v;
    }
  };

  // the wave's Q fragments (rows past q_len read row q_len - 1, the wave's own last row; their outputs are
  // never stored).  O is written over Q: each wave reads only its own rows, before it writes them.
  u32x4_t qf[4] = {};
  if (active) {
    const uint16_t* qrow = a.q + ((int64_t)b * a.q_len + min(qi, a.q_len - 1)) * D + h * 64 + hf * 8;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const u32x4_t*>(qrow + c * 16);
  }
  int kofs[4], vofs[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) kofs[c] = ((2 * c + hf) ^ ((fr >> 1) & 7)) << 4;
#pragma unroll
  for (int c2 = 0; c2 < 2; ++c2) vofs[c2] = ((2 * c2 + hf) ^ ((fr >> 2) & 3)) << 4;

  f32x16_t o[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) { o[0][e] = 0.0f; o[1][e] = 0.0f; }
  // m: the shift of the exponentials (log2 units), shared by the two lanes of a query, raised by
  // attn_tile_softmax only when the exponentials grow past 2^16 (the normalised output does not depend on
  // it); l: this lane's share of the softmax denominator
  float m = -INFINITY, l = 0.0f;

  cload(0);
  cstore(0, 0);
  __syncthreads();
  for (int c = 0; c < nchunks; ++c) {
    const int buf = c & 1, cb = c * kStreamKeys;
    if (c + 1 < nchunks) cload(cb + kStreamKeys);
    if (cb < w_end) {
      const char* kp = sbuf[buf] + fr * 128;
      const char* vp0 = sbuf[buf] + kStreamKeys * 128 + fr * 128;
      const char* vp1 = vp0 + 32 * 128;
      for (int j0 = 0; j0 < kStreamKeys && cb + j0 < w_end; j0 += 32) {
        u32x4_t kf[4], vf[4];
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) kf[cc] = *reinterpret_cast<const u32x4_t*>(kp + j0 * 128 + kofs[cc]);
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          vf[2 * c2] = *reinterpret_cast<const u32x4_t*>(vp0 + j0 * 2 + vofs[c2]);
          vf[2 * c2 + 1] = *reinterpret_cast<const u32x4_t*>(vp1 + j0 * 2 + vofs[c2]);
        }
        // S^T[key][q] = K . Q^T; s[e] is key cb + j0 + 16*(e/8) + hf*8 + e%8
        f32x16_t s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) s = mfma32x32x16(kf[cc], qf[cc], s);
        const int jg = cb + j0;
        if (jg + 31 > qi0 + off || jg + 32 > a.kv) {  // some key of the tile is masked for some query
          const int r = lim - jg;
#pragma unroll
          for (int e = 0; e < 16; ++e) s[e] = (16 * (e >> 3) + (e & 7) <= r) ? s[e] : -INFINITY;
        }
        uint32_t pk[8];
        // max first: the lazy form needs about 14 more registers than the 128 of four waves per SIMD
        const float ps = attn_tile_softmax<false>(s, a.scale_log2, m, l, o, pk);
        l += ps;
        // O^T[d][q] += V^T . P^T; chunk c2 of P^T holds keys j0 + 16*c2 + hf*8 + 0..7
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          const u32x4_t pb = {pk[4 * c2], pk[4 * c2 + 1], pk[4 * c2 + 2], pk[4 * c2 + 3]};
          o[0] = mfma32x32x16(vf[2 * c2], pb, o[0]);
          o[1] = mfma32x32x16(vf[2 * c2 + 1], pb, o[1]);
        }
      }
    }
    if (c + 1 < nchunks) cstore(cb + kStreamKeys, buf ^ 1);
    __syncthreads();
  }
  if (!active) return;
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (qi < a.q_len) {
    const float inv = 1.0f / l;
    uint16_t* orow = a.o + ((int64_t)b * a.q_len + qi) * D + h * 64;
    // o[db][e] is d = db*32 + (e/4)*8 + hf*4 + e%4
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + g * 8 + hf * 4;
        u32x2_t w;
        w[0] = pack_bf16x2(o[db][4 * g] * inv, o[db][4 * g + 1] * inv);
        w[1] = pack_bf16x2(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv);
        *reinterpret_cast<u32x2_t*>(orow + d) = w;
      }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct BlockLayout {
  int64_t h = 0, q = 0, k = 0, vt = 0, g = 0, total = 0;
  int kv_pad = 0;  // keys of a head held by the attention (kv rounded up to 32)
  int vt_ld = 0;   // V^T row stride (kv rounded up to 64: rows start on 128-byte lines)
};

static int64_t align256(int64_t v) { return (v + 255) & ~int64_t(255); }

// d_model 128, and 256 above kFusedMinRows kept rows, run the out-projection, RMSNorm2 and the FFN in one kernel, whose
// tiles of 128 rows walk the whole hidden dimension one after another: 50 us at d_model 256 however few rows there are,
// 53 us for 17,408 rows, 81 us for 34,816.  Below, and at d_model 384 / 512 (whose rows do not fit its registers), three
// kernels split that work over the chip: 30 us for 4,352 rows, 57 us for 17,408, 112 us for 34,816.  (Those are for a
// hidden dimension of 1,024; from 128 to 4,096 hidden units and 0 to 64 NS tokens, blocks of 256 to 13,952 rows took at
// most 0.98 of their time with the one kernel and the weight-stationary projection.  At d_model 128 the one kernel is the
// faster at every size: 1 sample 43 against 49 us per block.)  The three keep the GELU activations (g) in the workspace,
// and RMSNorm2's rows (h) for a caller that asks for them.
// The residual GEMM reaches the rows of g within 2^32 bytes, so d_model 256 takes the three only where all of g lies in them.
constexpr int64_t kFusedMinRows = 14000;
static int64_t split_max_rows(const pdm_block_desc& d) {  // kept rows up to which the three kernels run
  if (d.d_model == 128) return 0;
  return d.d_model == 256 ? std::min(kFusedMinRows, ((int64_t(1) << 31) - 1) / d.ffn_dim) : INT64_MAX;
}
static bool fused_path(const pdm_block_desc& d) { return (int64_t)d.batch * d.q_len > split_max_rows(d); }
// Kept rows for which the workspace holds h and g.  At d_model 256 that is the largest batch the three kernels take,
// also when this one is larger, so that a workspace sized for one batch is enough for every smaller one.
static int64_t split_rows(const pdm_block_desc& d) { return std::min((int64_t)d.batch * d.q_len, split_max_rows(d)); }
// d_model 256: rows of x from which the weight-stationary Q/K/V projection (384 KB of weight into every CU's registers
// first: 34 us however few rows) is faster than the streaming one.  Per block: 6,400 rows 34 against 14 us, 51,200 rows
// 62 against 49 us, 102,400 rows 277 against 274 us (whole block), 204,800 rows 448 against 461 us (whole block).
constexpr int64_t kQkvStationaryMinRows = 120000;

// room: with space for h and g wherever split_rows asks for it; without it a d_model 256 block runs the fused FFN
// whatever its rows, so that a workspace of Q, K and V^T is enough at any size.
static BlockLayout block_layout(const pdm_block_desc& d, bool room = true) {
  BlockLayout L;
  const int64_t B = d.batch, D = d.d_model;
  L.kv_pad = (d.kv_len + 31) & ~31;
  L.vt_ld = (d.kv_len + 63) & ~63;
  int64_t off = 0;
  L.q = off; off = align256(off + B * d.q_len * D * 2);                 // Q, later attention output
  L.k = off; off = align256(off + B * d.kv_len * D * 2);                // K
  L.vt = off; off = align256(off + B * (D / 64) * 64 * (int64_t)L.vt_ld * 2);  // V^T per head
  const int64_t rows = room || d.d_model > 256 ? split_rows(d) : 0;
  L.h = off; off = align256(off + rows * D * 2);                        // RMSNorm2 rows
  L.g = off; off = align256(off + rows * (int64_t)d.ffn_dim * 2);       // GELU(FFN-up)
  L.total = off;
  return L;
}

static const char* check_desc(const pdm_block_desc* d) {
  if (!d) return "null desc";
  if (d->batch < 1) return "batch must be >= 1";
  if (d->d_model < 128 || d->d_model > 512 || d->d_model % 128) return "d_model must be 128, 256, 384 or 512";
  if (d->n_heads * 64 != d->d_model) return "head dim must be 64 (n_heads = d_model / 64)";
  if (d->ffn_dim < 128 || d->ffn_dim % 128) return "ffn_dim must be a positive multiple of 128";
  if (d->n_ns < 0) return "n_ns must be >= 0";
  if (!(d->n_ns <= d->q_len && d->q_len <= d->kv_len)) return "need n_ns <= q_len <= kv_len";
  if (d->q_len < 1) return "q_len must be >= 1";
  return nullptr;
}

// Row tiles of rows_per_tile rows: the shared group's tiles, then tiles_b per NS token.
static int64_t row_tiles(GemmArgs& g, int rows_per_tile) {
  g.tiles_s = (int)(((int64_t)g.B * g.n_s + rows_per_tile - 1) / rows_per_tile);
  g.tiles_b = (g.B + rows_per_tile - 1) / rows_per_tile;
  return (int64_t)g.tiles_s + (int64_t)g.n_ns * g.tiles_b;
}

// Two workgroups of four waves per CU walk the row tiles of the fused FFN.
static int launch_ffn(GemmArgs& g, int D, hipStream_t s) {
  constexpr int NW = 4, WPS = 2;
  const int64_t tiles = row_tiles(g, NW * 32);
  if (tiles == 0) return PDM_OK;
  PDM_CHECK_ARG(tiles < (int64_t(1) << 31), "FFN grid too large");
  g.total_blocks = tiles;
  static std::once_flag once[64];
  static hipError_t err[64];
  static int ncu[64];
  int dev = 0;
  PDM_CHECK_HIP(hipGetDevice(&dev));
  PDM_CHECK_ARG(dev >= 0 && dev < 64, "device index out of range");
  std::call_once(once[dev], [&] { err[dev] = hipDeviceGetAttribute(&ncu[dev], hipDeviceAttributeMultiprocessorCount, dev); });
  PDM_CHECK_HIP(err[dev]);
  const int64_t grid = std::min<int64_t>(tiles, (int64_t)std::max(ncu[dev], 1) * WPS);
  if (D == 256) hipLaunchKernelGGL((ffn_kernel<256, NW, WPS>), dim3((unsigned)grid), dim3(NW * 64), 0, s, g);
  else hipLaunchKernelGGL((ffn_kernel<128, NW, WPS>), dim3((unsigned)grid), dim3(NW * 64), 0, s, g);
  PDM_CHECK_LAUNCH();
  return PDM_OK;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Largest LDS footprint of attn_lds_kernel; longer sequences run attn_stream_kernel,
// which streams K and V^T through LDS in chunks.
constexpr int64_t kAttnLdsMax = (int64_t)kAttnLdsMaxKeys * 256;
// LDS of one workgroup on gfx950: K, V^T and, when it fits, the head's Q
constexpr int64_t kAttnLdsLimit = 160 * 1024;

// Launches attn_lds_kernel<NP, NW> on a persistent grid: as many workgroups as
// fit on the device at once, each walking (sample, head) pairs.  The LDS limit
// is raised above the default 64 KiB once per process, device and instance.
template <int NP, int NW>
static int launch_attn_lds(AttnArgs aa, int64_t lds, hipStream_t s) {
  static std::once_flag once[64];
  static hipError_t err[64];
  static int ncu[64];
  int dev = 0;
  PDM_CHECK_HIP(hipGetDevice(&dev));
  PDM_CHECK_ARG(dev >= 0 && dev < 64, "device index out of range");
  std::call_once(once[dev], [&] {
    err[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_lds_kernel<NP, NW>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kAttnLdsLimit);
    if (err[dev] == hipSuccess) err[dev] = hipDeviceGetAttribute(&ncu[dev], hipDeviceAttributeMultiprocessorCount, dev);
  });
  PDM_CHECK_HIP(err[dev]);
  // the copy rounds must cover the kv_pad K rows (NW * 8 per round) and the kv_pad / 8 pieces of each of the
  // 64 V^T rows (8 pieces of NW * 8 rows per round)
  constexpr int RPR = NW * 8;
  PDM_CHECK_ARG(aa.kv_pad <= RPR * NP && aa.kv_pad / 8 <= 8 * (NP / (64 / RPR)), "attention copy rounds too few");
  int per_cu = 0;
  PDM_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, attn_lds_kernel<NP, NW>, NW * 64, (size_t)lds));
  const int64_t bh = (int64_t)aa.B * aa.H;
  PDM_CHECK_ARG(bh < (int64_t(1) << 31), "batch * heads too large");
  int64_t grid = std::min<int64_t>(bh, (int64_t)std::max(ncu[dev], 1) * std::max(per_cu, 1));
  // Few heads leave CUs idle while a head's waves share four SIMDs: up to four workgroups then share its query tiles,
  // each with its own copy of K and V^T (Q straight from memory).  1 / 2 / 4 workgroups per head, stacks in us:
  // 4 layers d 256, B = 16 (64 heads, 9 tiles) 200.7 / 194.8 / 187.5; 3 layers d 256, B = 1, 596 keys 160.6 / 139.4 /
  // 134.7, d 128, B = 60, 596 keys (120 heads, so two) 203.7 / 179.2; eight were no faster than four.
  aa.parts = 1;
  if (NW == 8) {
    const int64_t tiles = (aa.q_len + 31) / 32;
    aa.parts = (int)std::max<int64_t>(1, std::min<int64_t>({4, tiles, (int64_t)std::max(ncu[dev], 1) / bh}));
  }
  if (aa.parts > 1) {
    aa.q_lds = 0;
    grid = bh * aa.parts;
  }
  hipLaunchKernelGGL((attn_lds_kernel<NP, NW>), dim3((unsigned)grid), dim3(NW * 64), (unsigned)lds, s, aa);
  PDM_CHECK_LAUNCH();
  return PDM_OK;
}

}  // namespace pdm

using namespace pdm;

extern "C" int64_t pdm_onetrans_block_workspace_size(const pdm_block_desc* desc) {
  clear_error();
  if (const char* e = check_desc(desc)) {
    set_error(std::string("pdm_onetrans_block_workspace_size: ") + e);
    return PDM_ERR_INVALID;
  }
  return block_layout(*desc).total;
}

namespace pdm {

// One block on stream s; the descriptor is checked, the pointers are not.  room: as block_layout's.
static int block_fwd(const pdm_block_desc& d, const float* x, const pdm_block_weights* w, float* y, void* workspace,
                     bool room, hipStream_t s) {
  const BlockLayout L = block_layout(d, room);
  const bool fused = fused_path(d) || (d.d_model == 256 && !room);
  char* ws = reinterpret_cast<char*>(workspace);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + L.h);
  uint16_t* q = reinterpret_cast<uint16_t*>(ws + L.q);
  uint16_t* k = reinterpret_cast<uint16_t*>(ws + L.k);
  uint16_t* vt = reinterpret_cast<uint16_t*>(ws + L.vt);
  uint16_t* g = reinterpret_cast<uint16_t*>(ws + L.g);
  const int B = d.batch, D = d.d_model, H = d.n_heads, F = d.ffn_dim;
  const int kv = d.kv_len, ql = d.q_len, nns = d.n_ns;
  int st;

  if (D == 256 && (int64_t)B * kv > kQkvStationaryMinRows) {
    // 1. Q (tail rows), K, V^T = RMSNorm1(x) . Wqkv^T  (weight-stationary, norm fused)
    QkvArgs qa{};
    qa.x = x; qa.x_bstride = (int64_t)kv * D; qa.norm_w = w->norm1_w;
    qa.W = reinterpret_cast<const uint16_t*>(w->s_qkv_w);
    qa.W_ns = reinterpret_cast<const uint16_t*>(w->ns_qkv_w);
    qa.q = q; qa.k = k; qa.vt = vt;
    qa.B = B; qa.kv = kv; qa.q_len = ql; qa.n_ns = nns; qa.kv_pad = L.vt_ld;
    if ((st = launch_qkv_stationary(qa, D, s)) != PDM_OK) return st;
  } else {
    // 1. Q (tail rows), K, V^T = RMSNorm1(x) . Wqkv^T  (norm fused)
    RowProjArgs r0{};
    r0.x = x; r0.in_bstride = (int64_t)kv * D; r0.norm_w = w->norm1_w;
    r0.W = reinterpret_cast<const uint16_t*>(w->s_qkv_w);
    r0.W_ns = reinterpret_cast<const uint16_t*>(w->ns_qkv_w);
    r0.B = B; r0.n_s = kv - nns; r0.n_ns = nns; r0.N = 3 * D;
    r0.q = q; r0.k = k; r0.vt = vt; r0.kv = kv; r0.q_len = ql; r0.kv_pad = L.vt_ld;
    if ((st = launch_row_proj(r0, D, ROWPROJ_QKV, s)) != PDM_OK) return st;
  }
  // 2. attention -> O (written over Q: each wave reads its Q rows before writing them)
  {
    AttnArgs aa{};
    aa.q = q; aa.k = k; aa.vt = vt; aa.o = q;
    aa.B = B; aa.H = H; aa.q_len = ql; aa.kv = kv; aa.kv_pad = L.kv_pad; aa.vt_ld = L.vt_ld;
    aa.scale_log2 = 1.4426950408889634f / 8.0f;
    const int64_t gy = (int64_t)B * H;
    const int64_t lds = (int64_t)L.kv_pad * 256;  // K rows (128 B) + V^T rows (2 B per key) of one head
    if (lds <= kAttnLdsMax) {
      const int np = (L.kv_pad * 8 + 511) / 512;      // copy rounds of 8 waves
      const int np4 = 2 * ((L.kv_pad + 63) / 64);      // and of 4 (two rounds per 64 keys of V^T)
      if ((ql + 31) / 32 <= 4 && np4 <= 8) {
        // at most 4 query tiles per head: workgroups of 4 waves, two per CU on two heads
        if (np4 <= 2) st = launch_attn_lds<2, 4>(aa, lds, s);
        else if (np4 <= 4) st = launch_attn_lds<4, 4>(aa, lds, s);
        else if (np4 <= 6) st = launch_attn_lds<6, 4>(aa, lds, s);
        else st = launch_attn_lds<8, 4>(aa, lds, s);
      } else {
        // 8 waves: with at most 16 query tiles (two per wave) and room in LDS, Q is staged there too
        const int64_t lds_q = lds + (int64_t)((ql + 31) / 32) * 32 * 128;
        aa.q_lds = (ql + 31) / 32 <= 16 && lds_q <= kAttnLdsLimit;
        const int64_t lds8 = aa.q_lds ? lds_q : lds;
        if (np <= 2) st = launch_attn_lds<2, 8>(aa, lds8, s);
        else if (np <= 4) st = launch_attn_lds<4, 8>(aa, lds8, s);
        else if (np <= 7) st = launch_attn_lds<7, 8>(aa, lds8, s);
        else st = launch_attn_lds<(kAttnLdsMaxKeys * 8 + 511) / 512, 8>(aa, lds8, s);
      }
      if (st != PDM_OK) return st;
    } else {
      // keys streamed through LDS in chunks, 8 waves (256 queries) per workgroup
      constexpr int kNW = PDM_ATTN_STREAM_NW;
      const int n_qb = (ql + 32 * kNW - 1) / (32 * kNW);
      const int64_t n_items = gy * n_qb;
      PDM_CHECK_ARG(n_items < (int64_t(1) << 31), "batch * heads * query blocks must be < 2^31");
      hipLaunchKernelGGL(attn_stream_kernel<kNW>, dim3((unsigned)n_items), dim3(kNW * 64), 0, s, aa, n_qb, n_items);
    }
    PDM_CHECK_LAUNCH();
  }
  if (fused) {
    // 3. z = bf16(O . Wout^T) + x[:, kv - q_len:], y = z + W2 . gelu(W1 . RMSNorm2(z)):
    // out-projection, norm, both FFN GEMMs and GELU in one kernel
    GemmArgs g2{};
    g2.A = q; g2.a_bstride = (int64_t)ql * D;
    g2.Wo = reinterpret_cast<const uint16_t*>(w->out_w);
    g2.res = x; g2.res_bstride = (int64_t)kv * D; g2.res_toff = kv - ql;
    g2.norm_w = w->norm2_w;
    g2.W = reinterpret_cast<const uint16_t*>(w->s_w1);
    g2.W_ns = reinterpret_cast<const uint16_t*>(w->ns_w1);
    g2.W2 = reinterpret_cast<const uint16_t*>(w->s_w2);
    g2.W2_ns = reinterpret_cast<const uint16_t*>(w->ns_w2);
    g2.B = B; g2.n_s = ql - nns; g2.n_ns = nns; g2.N = F; g2.K = D;
    g2.out = y; g2.out_bstride = (int64_t)ql * D;
    return launch_ffn(g2, D, s);
  }
  // 3. z = bf16(O . Wout^T) + x[:, kv - q_len:]  -> y
  {
    ResidArgs g1{};
    g1.round_bf16 = 1;
    g1.A = q; g1.a_bstride = (int64_t)ql * D;
    g1.W = reinterpret_cast<const uint16_t*>(w->out_w);
    g1.B = B; g1.n_s = ql; g1.n_ns = 0; g1.N = D; g1.K = D;
    g1.out = y; g1.out_bstride = (int64_t)ql * D;
    g1.res = x; g1.res_bstride = (int64_t)kv * D; g1.res_toff = kv - ql;
    if ((st = launch_resid_gemm(g1, s)) != PDM_OK) return st;
  }
  // 4. g = bf16(gelu(bf16(RMSNorm2(z) . W1^T)))  [B, q_len, F]; RMSNorm2(z) itself only on request, nothing here reads it
  {
    RowProjArgs r2{};
    r2.x = y; r2.norm_w = w->norm2_w; r2.in_bstride = (int64_t)ql * D;
    r2.W = reinterpret_cast<const uint16_t*>(w->s_w1);
    r2.W_ns = reinterpret_cast<const uint16_t*>(w->ns_w1);
    r2.B = B; r2.n_s = ql - nns; r2.n_ns = nns; r2.N = F;
    r2.h = (d.flags & PDM_BLOCK_KEEP_NORM2) ? h : nullptr; r2.out = g; r2.out_bstride = (int64_t)ql * F;
    if ((st = launch_row_proj(r2, D, ROWPROJ_GELU, s)) != PDM_OK) return st;
  }
  // 5. y = z + g . W2^T
  {
    ResidArgs g3{};
    g3.A = g; g3.a_bstride = (int64_t)ql * F;
    g3.W = reinterpret_cast<const uint16_t*>(w->s_w2);
    g3.W_ns = reinterpret_cast<const uint16_t*>(w->ns_w2);
    g3.B = B; g3.n_s = ql - nns; g3.n_ns = nns; g3.N = D; g3.K = F;
    g3.out = y; g3.out_bstride = (int64_t)ql * D;
    g3.res = y; g3.res_bstride = (int64_t)ql * D; g3.res_toff = 0;
    if ((st = launch_resid_gemm(g3, s)) != PDM_OK) return st;
  }
  return PDM_OK;
}

// Checks the weight pointers of one layer (alignment of every tensor the kernels read with 16-byte loads).
static int check_block_weights(const pdm_block_desc& d, const pdm_block_weights* w) {
  PDM_CHECK_ARG(w, "null weights");
  PDM_CHECK_ARG(w->norm1_w && w->s_qkv_w && w->out_w && w->norm2_w && w->s_w1 && w->s_w2, "null weight pointer");
  PDM_CHECK_ARG(d.n_ns == 0 || (w->ns_qkv_w && w->ns_w1 && w->ns_w2), "null per-token weight pointer");
  const void* ptrs[] = {w->s_qkv_w, w->out_w, w->s_w1, w->s_w2, d.n_ns ? w->ns_qkv_w : w->s_qkv_w,
                        d.n_ns ? w->ns_w1 : w->s_w1, d.n_ns ? w->ns_w2 : w->s_w2, w->norm1_w, w->norm2_w};
  for (const void* p : ptrs) PDM_CHECK_ARG(aligned16(p), "every tensor must be 16-byte aligned");
  return PDM_OK;
}

}  // namespace pdm

extern "C" int pdm_onetrans_block_fwd(const pdm_block_desc* desc, const float* x, const pdm_block_weights* w,
                                      float* y, void* workspace, int64_t workspace_bytes, pdm_stream_t stream) {
  clear_error();
  if (const char* e = check_desc(desc)) {
    set_error(std::string("pdm_onetrans_block_fwd: ") + e);
    return PDM_ERR_INVALID;
  }
  const pdm_block_desc& d = *desc;
  PDM_CHECK_ARG(x && w && y && workspace, "null pointer");
  int st;
  if ((st = check_block_weights(d, w)) != PDM_OK) return st;
  const int64_t need = block_layout(d).total;
  const bool room = workspace_bytes >= need;
  if (!room && workspace_bytes < block_layout(d, false).total) {
    set_error("pdm_onetrans_block_fwd: workspace of " + std::to_string(workspace_bytes) + " bytes, need " +
              std::to_string(need));
    return PDM_ERR_WORKSPACE;
  }
  PDM_CHECK_ARG(aligned16(x) && aligned16(y) && aligned16(workspace), "every tensor must be 16-byte aligned");
  PDM_CHECK_ARG((const void*)y != (const void*)x, "y must not alias x");
  return block_fwd(d, x, w, y, workspace, room, reinterpret_cast<hipStream_t>(stream));
}

// ---------------------------------------------------------------------------
// Block stack: the layer loop of OneTransModel._backbone.  Layer l runs on the
// previous layer's output (kv_len = its q_len) and keeps q_s[l] + n_ns tokens.
// Workspace: one block workspace sized for the largest layer, reused by every
// layer, then the fp32 outputs of the inner layers in two alternating buffers
// of the largest inner layer's size.
// ---------------------------------------------------------------------------
namespace pdm {

struct StackLayout {
  int64_t block;    // bytes of the shared block workspace
  int64_t buf[2];   // offsets of the two inner-layer output buffers
  int64_t total;
};

static const char* stack_layout(const pdm_block_desc* desc, const int32_t* q_s, int32_t n_layers, StackLayout& S,
                                bool room = true) {
  if (!desc) return "null desc";
  if (!q_s) return "null q_s";
  if (n_layers < 1 || n_layers > PDM_STACK_MAX_LAYERS) return "n_layers must be in [1, PDM_STACK_MAX_LAYERS]";
  pdm_block_desc d = *desc;
  int64_t block = 0, inner = 0;
  for (int l = 0; l < n_layers; ++l) {
    if (q_s[l] < 0) return "q_s must be >= 0";
    d.q_len = q_s[l] + desc->n_ns;
    if (const char* e = check_desc(&d)) return e;
    block = std::max(block, block_layout(d, room).total);
    if (l + 1 < n_layers) inner = std::max(inner, align256((int64_t)d.batch * d.q_len * d.d_model * 4));
    d.kv_len = d.q_len;
  }
  S.block = align256(block);
  S.buf[0] = S.block;
  S.buf[1] = S.block + (n_layers > 1 ? inner : 0);
  S.total = S.buf[1] + (n_layers > 2 ? inner : 0);
  return nullptr;
}

}  // namespace pdm

extern "C" int64_t pdm_onetrans_stack_workspace_size(const pdm_block_desc* desc, const int32_t* q_s,
                                                     int32_t n_layers) {
  clear_error();
  StackLayout S;
  if (const char* e = stack_layout(desc, q_s, n_layers, S)) {
    set_error(std::string("pdm_onetrans_stack_workspace_size: ") + e);
    return PDM_ERR_INVALID;
  }
  return S.total;
}

extern "C" int pdm_onetrans_stack_fwd(const pdm_block_desc* desc, const int32_t* q_s, int32_t n_layers,
                                      const float* x, const pdm_block_weights* weights, float* y, void* workspace,
                                      int64_t workspace_bytes, pdm_stream_t stream) {
  clear_error();
  StackLayout S;
  if (const char* e = stack_layout(desc, q_s, n_layers, S)) {
    set_error(std::string("pdm_onetrans_stack_fwd: ") + e);
    return PDM_ERR_INVALID;
  }
  PDM_CHECK_ARG(x && weights && y && workspace, "null pointer");
  const int64_t need = S.total;
  const bool room = workspace_bytes >= need;
  if (!room) stack_layout(desc, q_s, n_layers, S, false);
  if (workspace_bytes < S.total) {
    set_error("pdm_onetrans_stack_fwd: workspace of " + std::to_string(workspace_bytes) + " bytes, need " +
              std::to_string(need));
    return PDM_ERR_WORKSPACE;
  }
  PDM_CHECK_ARG(aligned16(x) && aligned16(y) && aligned16(workspace), "every tensor must be 16-byte aligned");
  PDM_CHECK_ARG((const void*)y != (const void*)x, "y must not alias x");
  pdm_block_desc d = *desc;
  int st;
  for (int l = 0; l < n_layers; ++l)
    if ((st = check_block_weights(d, &weights[l])) != PDM_OK) return st;
  auto s = reinterpret_cast<hipStream_t>(stream);
  char* ws = reinterpret_cast<char*>(workspace);
  const float* in = x;
  for (int l = 0; l < n_layers; ++l) {
    d.q_len = q_s[l] + desc->n_ns;
    float* out = l + 1 == n_layers ? y : reinterpret_cast<float*>(ws + S.buf[l & 1]);
    if ((st = block_fwd(d, in, &weights[l], out, ws, room, s)) != PDM_OK) return st;
    in = out;
    d.kv_len = d.q_len;
  }
  return PDM_OK;
}
