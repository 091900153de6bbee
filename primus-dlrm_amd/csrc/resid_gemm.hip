// Residual projections of the OneTrans block: out = A . W^T + res for bf16 rows of K columns.  The out-projection
// (K = d_model) rounds the product to bf16 as autocast does; the FFN-down (K = ffn_dim) adds it in fp32, as the fused
// FFN kernel does, at most half a bf16 step of the FFN output away from autocast.
//
// Tiles of TM rows x TN columns, four waves.  The rows and the weight stream through an LDS ring of BK-column stages
// filled by LDS DMA, NST - 1 stages ahead, one barrier per stage; the addresses are one 32-bit offset per lane and row
// plus a scalar base.  Two workgroups share a CU with independent barriers, so one's first stages, residual reads and
// stores run beside the other's MFMAs.  Rows are (sample, token) pairs: S tokens flattened over the samples use the
// shared weight, every NS token has row tiles of its own with its own weight; rows past the end read the tile's last
// row again and are not stored.
#include <algorithm>

#include "pdm_common.h"
#include "mfma_common.h"
#include "block_kernels.h"

namespace pdm {

// WM x WN waves, each (TM / WM) x (TN / WN) outputs in 32 x 32 MFMA blocks
template <int TM, int TN, int WM, int BK, int NST>
__global__ __launch_bounds__(256, 2) void resid_gemm_kernel(ResidArgs a) {
  constexpr int WN = 4 / WM, MB = TM / WM / 32, NB = TN / WN / 32;
  constexpr int PF = NST - 1, RB = BK * 2;     // stages ahead, bytes per row of a stage
  constexpr int LPR = BK / 8;                  // lanes (16-byte pieces) per row
  constexpr int STAGE = (TM + TN) * RB;
  constexpr int NA = TM * RB / 4096, NW = TN * RB / 4096;  // DMA instructions per wave and stage
  static_assert(NA * 4096 == TM * RB && NW * 4096 == TN * RB, "a stage splits evenly over the waves");
  constexpr int SROW = NB * 128 + 16;          // epilogue: LDS bytes per staged output row
  constexpr int LDS = NST * STAGE > 4 * 32 * SROW ? NST * STAGE : 4 * 32 * SROW;
  __shared__ __attribute__((aligned(256))) char lds[LDS];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;

  // workgroup -> (row tile, column tile); the column tiles of a row tile are neighbours on one XCD (workgroups go to
  // the 8 XCDs in turn), whose L2 serves the rows to all of them.  The NS tiles come first.
  const int nt = a.N / TN;
  const int n_ns_wgs = a.n_ns * a.tiles_b * nt, n_s_wgs = a.tiles_s * nt;
  const bool is_s = (int)blockIdx.x >= n_ns_wgs;
  int rest = is_s ? (int)blockIdx.x - n_ns_wgs : (int)blockIdx.x;
  const int full = (is_s ? n_s_wgs : n_ns_wgs) & ~7;
  if (rest < full) rest = (rest & 7) * (full >> 3) + (rest >> 3);
  const int mt = rest / nt, n0 = (rest - mt * nt) * TN;
  const int g = is_s ? 0 : mt / a.tiles_b;
  const int64_t r0 = is_s ? (int64_t)mt * TM : (int64_t)(mt - g * a.tiles_b) * TM;  // the tile's first row
  const int64_t nrows = is_s ? (int64_t)a.B * a.n_s : a.B;
  const int rows = (int)min((int64_t)TM, nrows - r0);
  const int b0 = is_s ? (int)(r0 / a.n_s) : (int)r0, t0 = is_s ? (int)(r0 - (int64_t)b0 * a.n_s) : a.n_s + g;
  // row i of the tile: sample b0 + db, token t
  auto row_of = [&](int i, int& db, int& t) {
    if (is_s) {
      const uint32_t u = (uint32_t)(t0 + i);
      db = (int)(u / (uint32_t)a.n_s);
      t = (int)(u - (uint32_t)db * (uint32_t)a.n_s);
    } else {
      db = i;
      t = t0;
    }
  };
  const uint16_t* W = (is_s ? a.W : a.W_ns + (int64_t)g * a.N * a.K) + (int64_t)n0 * a.K;
  const uint64_t abase = (uint64_t)(uintptr_t)(a.A + (int64_t)b0 * a.a_bstride), wbase = (uint64_t)(uintptr_t)W;

  // DMA instruction p of a wave fills 64 / LPR rows; piece v of row r lies at slot v ^ swz(r), which spreads the 32
  // rows of a fragment read over the banks
  auto swz = [](int r) { return BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; };
  uint32_t aoff[NA], woff[NW];
#pragma unroll
  for (int p = 0; p < NA; ++p) {
    const int r = (wave * NA + p) * (64 / LPR) + lane / LPR;
    int db, t;
    row_of(min(r, rows - 1), db, t);
    aoff[p] = (uint32_t)(((int64_t)db * a.a_bstride + (int64_t)t * a.K) * 2) + (((lane % LPR) ^ swz(r)) << 4);
  }
#pragma unroll
  for (int p = 0; p < NW; ++p) {
    const int r = (wave * NW + p) * (64 / LPR) + lane / LPR;
    woff[p] = (uint32_t)r * a.K * 2 + (((lane % LPR) ^ swz(r)) << 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  auto dma = [&](int kt, int stg) {
    const uint64_t k2 = (uint64_t)kt * RB;
#pragma unroll
    for (int p = 0; p < NA; ++p) lds_dma16(abase + k2, aoff[p], lds0 + stg * STAGE + (wave * NA + p) * 1024);
#pragma unroll
    for (int p = 0; p < NW; ++p) lds_dma16(wbase + k2, woff[p], lds0 + stg * STAGE + TM * RB + (wave * NW + p) * 1024);
  };

  f32x16_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int nk = a.K / BK;
#pragma unroll
  for (int j = 0; j < PF; ++j) dma(min(j, nk - 1), j);
  // fragment (row block, k step s): lane row fr, piece 2 s + hf
  const uint32_t fa = (uint32_t)((wm * MB * 32 + fr) * RB + ((hf ^ swz(fr)) << 4));
  const uint32_t fw = (uint32_t)(TM * RB + (wn * NB * 32 + fr) * RB + ((hf ^ swz(fr)) << 4));
  int stg = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // loads complete in issue order: stage kt has landed once only the PF - 1 later stages' are outstanding
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((PF - 1) * (NA + NW)));
    __syncthreads();  // publishes every wave's part of the stage and frees stage kt - 1
    dma(min(kt + PF, nk - 1), stg == 0 ? NST - 1 : stg - 1);  // past the end: the last one again, read by nobody
    const uint32_t sb = lds0 + stg * STAGE;
    stg = stg + 1 == NST ? 0 : stg + 1;
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      u32x4_t af[MB], wf[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i)
        af[i] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>((sb + (fa ^ (s << 5))) + i * 32 * RB);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        wf[j] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>((sb + (fw ^ (s << 5))) + j * 32 * RB);
      // rows on lanes: acc[i][j] holds row i*32 + fr, columns j*32 + (e/4)*8 + hf*4 + e%4
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma32x32x16(wf[j], af[i], acc[i][j]);
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // no DMA may land in LDS once the epilogue uses it
  __syncthreads();

  // epilogue, 32 rows of the wave at a time: its NB * 32 columns pass through LDS, so that residual reads and stores
  // take whole row segments of NB * 128 bytes (NB * 8 lanes per row)
  constexpr int LR = NB * 8, RPI = 64 / LR;  // lanes per row, rows per instruction
  char* st = lds + wave * 32 * SROW;
  const int c4 = (lane % LR) * 4;
  const int col = n0 + wn * NB * 32 + c4;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    int64_t oo[32 / RPI];
    f32x4_t res[32 / RPI];
#pragma unroll
    for (int q = 0; q < 32 / RPI; ++q) {
      const int r = wm * MB * 32 + i * 32 + q * RPI + lane / LR;
      int db, t;
      row_of(min(r, rows - 1), db, t);
      res[q] = *reinterpret_cast<const f32x4_t*>(a.res + (int64_t)(b0 + db) * a.res_bstride + (int64_t)(t + a.res_toff) * a.N + col);
      oo[q] = r < rows ? (int64_t)(b0 + db) * a.out_bstride + (int64_t)t * a.N + col : -1;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4_t*>(st + fr * SROW + j * 128 + q * 32 + hf * 16) =
            a.round_bf16 ? f32x4_t{bf16_round(acc[i][j][4 * q]), bf16_round(acc[i][j][4 * q + 1]),
                                   bf16_round(acc[i][j][4 * q + 2]), bf16_round(acc[i][j][4 * q + 3])}
                         : f32x4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    // the wave's own LDS operations complete in order
#pragma unroll
    for (int q = 0; q < 32 / RPI; ++q) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(st + (q * RPI + lane / LR) * SROW + c4 * 4);
      if (oo[q] >= 0)
        *reinterpret_cast<f32x4_t*>(a.out + oo[q]) = f32x4_t{v.x + res[q].x, v.y + res[q].y, v.z + res[q].z, v.w + res[q].w};
    }
  }
}

template <int TM, int TN, int WM, int BK, int NST>
static int launch_tiles(ResidArgs a, hipStream_t s) {
  const int64_t tiles_s = ((int64_t)a.B * a.n_s + TM - 1) / TM;
  a.tiles_b = (a.B + TM - 1) / TM;
  const int64_t grid = (tiles_s + (int64_t)a.n_ns * a.tiles_b) * (a.N / TN);
  if (grid == 0) return PDM_OK;
  PDM_CHECK_ARG(grid < (int64_t(1) << 24), "GEMM grid too large");  // a launch dimension holds less than 2^32 threads
  // a tile's rows lie within 2^32 bytes of its first sample, and its weight rows of its first
  const int64_t samples = std::min<int64_t>(a.B, std::max(a.n_s ? (TM - 2) / a.n_s + 2 : 1, a.n_ns ? TM : 1));
  PDM_CHECK_ARG(samples * a.a_bstride * 2 < (int64_t(1) << 32), "GEMM rows too far apart");
  PDM_CHECK_ARG((int64_t)TN * a.K * 2 < (int64_t(1) << 32), "GEMM weight too large");
  a.tiles_s = (int)tiles_s;
  hipLaunchKernelGGL((resid_gemm_kernel<TM, TN, WM, BK, NST>), dim3((unsigned)grid), dim3(256), 0, s, a);
  PDM_CHECK_LAUNCH();
  return PDM_OK;
}

int launch_resid_gemm(const ResidArgs& a, hipStream_t s) {
  // Larger tiles read the rows and the weight fewer times, smaller ones fill the chip.  192 rows from four rounds of
  // workgroups on (OneTransL's second layer, B = 1024: out-projection 0.98, FFN-down 2.09 ms; 128 rows 1.04 and 2.24 ms;
  // 36,000 rows: 37 and 73 us against 34 and 67 us).  64 x 64 tiles with four stages below one 128 x 128 tile per CU
  // (400 tokens of d 384: a whole block 53 us, against 94 us with 256 x 128 tiles; 12,000 rows: 35 us against 31).
  auto tiles = [&](int tm, int tn) {
    return (((int64_t)a.B * a.n_s + tm - 1) / tm + (int64_t)a.n_ns * ((a.B + tm - 1) / tm)) * (a.N / tn);
  };
  if (tiles(192, 128) >= 4 * 512) return launch_tiles<192, 128, 2, 64, 2>(a, s);
  if (tiles(128, 128) >= 256) return launch_tiles<128, 128, 2, 64, 2>(a, s);
  return launch_tiles<64, 64, 2, 64, 4>(a, s);
}

}  // namespace pdm
