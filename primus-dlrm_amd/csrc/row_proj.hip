// Row projections of the OneTrans block: out = RMSNorm(x) . W^T for fp32 rows of D <= 512 columns, with the Q/K/V
// scatter or the GELU as the epilogue.
//
// Layout of the work.  A wave owns 32 rows and holds all D normalised columns of them in registers (the MFMA B
// operand: lane l has row l % 32, k = 8 (l / 32) .. +8 of every 16-wide step), so a row is read and normalised once
// whatever N is.  The weight streams through LDS in chunks of 32 output columns x D, filled by LDS DMA NST - 1 chunks
// ahead and shared by the workgroup's four waves.  Within a wave, the DMA of a later chunk and the epilogue of the
// previous one (rounding, GELU, stores) are issued between the MFMAs of the current chunk; two workgroups share a CU
// with independent barriers, so one's row loads run beside the other's MFMAs.
//
// A wave's rows are 32 consecutive tokens of ONE sample (S tokens, the shared weight) or one token of 32 samples (an NS
// token with its weight, or a last S token of every sample where few are left behind its whole blocks): addresses are a
// wave-uniform base plus row * stride, and a feature row of V^T receives runs of 8 tokens at multiples of 8.  Padding
// rows (the last block of a sample, samples past the batch) read the block's last row again and store nothing.
//
// What bounds it, at OneTransL's second layer (d 384, B = 1024, 1,552,384 rows in, 1,335,296 kept): the fp32 rows in and
// the bf16 outputs out (6.5 GB at the L2 for Q/K/V, 7.2 GB for FFN-up, 1.4 and 1.5 ms at a device copy's rate; 1.37 TFLOP,
// 0.55 ms of MFMA), behind them the vector instructions between the MFMAs (matrix units busy 43 and 44 %).  Q/K/V 1.70 ms
// against 0.63 (RMSNorm kernel) + 2.52 ms (128 x 256 LDS-tiled GEMM); FFN-up + GELU 1.97 ms against 0.53 + 2.61 ms.  What
// that took: addresses kept in registers and the GELU table reached by one shift (231 -> 144 vector instructions per
// chunk: 2.20 -> 2.00 ms), whole 64-byte segments per store, the NS tiles spread over the XCDs (2.14 -> 1.86 ms for
// Q/K/V), the normalised rows not stored (2.19 -> 1.97 ms for FFN-up).  64 rows per wave (half the LDS reads and weight
// traffic) need 192 operand registers and leave none to overlap the stores: 1.88 ms without the norm.
//
// Workgroups split the N columns of one row tile when there are few row tiles, so that a small batch fills the chip;
// the splits of a tile are neighbours on one XCD, whose L2 then serves the rows to all of them (4 layers of d 128 at
// B = 16: 186 -> 157 us with the splits).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "pdm_common.h"
#include "mfma_common.h"
#include "block_kernels.h"

namespace pdm {

// GELU table of this file: the top 2048 entries of mfma_common.h's range, |x| in (2^-13, 8].  Below it |x| is clamped
// to the first entry, where e differs from its value at |x| by less than 5e-5: x e and x (1 - e) both round to the
// bf16 value x / 2 (half a bf16 step is 2^-9 relative), so results are the longer table's bit for bit, and the table
// takes 8 KB: with the 72 KB ring of D = 384 two workgroups fill the 160 KB of LDS exactly.
constexpr uint32_t kGeluLo = GELU_T_HI - 2047u;
constexpr int kGeluN = 2048;

// g[0..3] = GELU of u[first .. first + 7], rounded to bf16 before and after; t: LDS address of the table.  The entry of
// a bf16 pattern is at byte 4 (pattern - kGeluLo), i.e. (fp32 bits >> 14) - 4 kGeluLo: one shift and an immediate.
__device__ __forceinline__ void gelu2048_pack(uint32_t t, const f32x16_t& u, int first, uint32_t* g) {
  float x[8], e[8];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const uint32_t p = pack_bf16x2(u[first + i], u[first + i + 1]);
    x[i] = __builtin_bit_cast(float, p << 16);
    x[i + 1] = __builtin_bit_cast(float, p & 0xffff0000u);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float c = __builtin_amdgcn_fmed3f(fabsf(x[i]), __builtin_bit_cast(float, kGeluLo << 16), 8.0f);
    e[i] = *reinterpret_cast<const __attribute__((address_space(3))) float*>((__builtin_bit_cast(uint32_t, c) >> 14) + (t - 4 * kGeluLo));
  }
#pragma unroll
  for (int i = 0; i < 8; i += 2)
    g[i >> 1] = pack_bf16x2(__builtin_fmaf(-fabsf(x[i]), e[i], fmaxf(x[i], 0.0f)),
                            __builtin_fmaf(-fabsf(x[i + 1]), e[i + 1], fmaxf(x[i + 1], 0.0f)));
}

// exchanges lanes 32..63 of a with lanes 0..31 of b
__device__ __forceinline__ void half_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// exchanges lanes 16..31 (48..63) of a with lanes 0..15 (32..47) of b
__device__ __forceinline__ void quarter_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// sum over the 16 lanes of a row, in every lane: the butterfly's additions (after each rotation the sums repeat with
// its period, so lane i - n holds what lane i ^ n does), without its trips through LDS
__device__ __forceinline__ float row16_sum(float v) {
  auto ror = [](float x, auto n) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 | decltype(n)::value, 0xf, 0xf, true));
  };
  v += ror(v, std::integral_constant<int, 8>{});
  v += ror(v, std::integral_constant<int, 4>{});
  v += ror(v, std::integral_constant<int, 2>{});
  v += ror(v, std::integral_constant<int, 1>{});
  return v;
}

// The 32 x 32 output tile whose line l % 32 (a row, or a feature of V^T) lies in lanes l and l + 32, packed to bf16
// (dword j of half h: outputs 16 h + 8 (j / 2) + 4 (l / 32) + 2 (j % 2) and the next), regrouped so that 16-byte
// stores write whole 64-byte segments: part 0 are lines 0..15, part 1 lines 16..31, lane l of part i holding
// outputs 8 piece .. 8 piece + 7 of line 16 i + l % 16, piece = 2 ((l / 16) % 2) + l / 32.
__device__ __forceinline__ void tile_segments(uint32_t (&p)[2][4]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    half_swap(p[h][0], p[h][2]);
    half_swap(p[h][1], p[h][3]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) quarter_swap(p[0][j], p[1][j]);
}

// 16-byte store at base + off (base wave-uniform), dropped for lanes with off == kNoStore: a buffer store whose range
// check discards them, so the instruction is always issued and the memory operations of a chunk can be counted.
constexpr uint32_t kNoStore = 0xFFFFFFFFu;
__device__ __forceinline__ void store16(void* base, uint32_t off, u32x4_t v) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7FFFFFFF, 0x00020000);
  __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)off, 0, 0);
}

// ring depth: as many 32-column chunks as two workgroups per CU leave room for, at most 4
template <int D>
constexpr int rowproj_stages() { return D <= 256 ? 4 : (D == 384 ? 3 : 2); }
template <int D>
constexpr int rowproj_lds(bool gelu) { return rowproj_stages<D>() * 64 * D + (gelu ? kGeluN * 4 : 0); }

template <int D, int EPI>
__global__ __launch_bounds__(256, 2) void rowproj_kernel(RowProjArgs a) {
  constexpr int KS = D / 16;          // MFMA k steps
  constexpr int NST = rowproj_stages<D>(), PF = NST - 1;
  constexpr int CHUNK = 64 * D;       // bytes of 32 weight rows
  constexpr int P = D / 8;            // 16-byte pieces per weight row
  constexpr int NDMA = P / 8;         // DMA instructions per wave and chunk: a wave fills 8 rows
  constexpr int LEAD = 4;             // weight fragments read ahead of their MFMA
  extern __shared__ __attribute__((aligned(16))) char lds[];
  float* gelu_t = reinterpret_cast<float*>(lds + NST * CHUNK);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int l16 = lane & 15, piece = 2 * ((lane >> 4) & 1) + hf;  // tile_segments

  // workgroup -> (row tile, column split): the token tiles first, then the S blocks, each group dealt so that neighbours
  // share an XCD (workgroups go to the 8 XCDs in turn).  The token tiles run sample by sample, all tokens of 128 samples
  // behind each other, so that the 2-byte V^T stores of neighbouring tokens meet in one L2 line (token by token, each
  // line went out from as many XCDs as it has NS tokens; 4,096 samples of 16 S and 16 NS tokens, whole block: d 128
  // 229 -> 162 us, d 384 1,295 -> 1,109; 8 NS tokens alone, d 128: 121 -> 88); every XCD then reads every token's
  // weight, which costs less.  With less than four tiles of samples, whose last may be nearly empty, they run token by
  // token, or the XCDs with the last tile would idle (130 samples of 17 S and 16 NS tokens, d 384: 85 against 81 us).
  // A tile's splits share its rows.
  // (With both groups in one such order the token tiles, the slowest, all fell to the last XCD.)
  const int n_tok_wgs = a.wgs_tok * a.split_tok;
  const bool is_s = (int)blockIdx.x >= n_tok_wgs;
  int rest = is_s ? (int)blockIdx.x - n_tok_wgs : (int)blockIdx.x;
  const int full = (is_s ? a.wgs_s * a.split_s : n_tok_wgs) & ~7;
  if (rest < full) rest = (rest & 7) * (full >> 3) + (rest >> 3);
  const int split = is_s ? a.split_s : a.split_tok;
  const int tile = rest / split, part = rest - tile * split;
  // the wave's rows: row i is (sample b0, token t0 + i) or (sample b0 + i, token t0)
  int b0, t0, rows;
  if (is_s) {
    const int64_t blk = (int64_t)tile * 4 + wave;
    b0 = (int)(blk / a.blocks_per_sample);
    t0 = (int)(blk - (int64_t)b0 * a.blocks_per_sample) * 32;
    rows = b0 < a.B ? min(32, a.n_blk - t0) : 0;
    if (b0 >= a.B) b0 = t0 = 0;
  } else {
    int st, g;
    if (a.tiles_b >= 4) {
      st = tile / a.n_tok;
      g = tile - st * a.n_tok;
    } else {
      g = tile / a.tiles_b;
      st = tile - g * a.tiles_b;
    }
    b0 = (st * 4 + wave) * 32;
    t0 = a.n_blk + g;
    rows = max(0, min(32, a.B - b0));
    if (rows == 0) b0 = 0;
  }
  const int last = max(rows - 1, 0);
  const uint16_t* W = t0 < a.n_s ? a.W : a.W_ns + (int64_t)(t0 - a.n_s) * a.N * D;

  const int nchunks = a.N / 32;
  const int c_begin = (int)((int64_t)nchunks * part / split), c_end = (int)((int64_t)nchunks * (part + 1) / split);

  // instruction p of the DMA of weight chunk c into ring stage stg: 16-byte piece v of row r lies at slot
  // v ^ (r & 15), so the 32 rows of a fragment read fall in distinct bank groups
  uint32_t doff[NDMA];
#pragma unroll
  for (int p = 0; p < NDMA; ++p) {
    const int o = p * 64 + lane, r = wave * 8 + o / P, v = (o % P) ^ (r & 15);
    doff[p] = (uint32_t)(r * (2 * D) + v * 16);
  }
  auto dma = [&](int c, int stg, int p) {
    lds_dma16((uint64_t)(uintptr_t)W + (uint64_t)c * CHUNK, doff[p],
              (uint32_t)(uintptr_t)(lds + stg * CHUNK + (wave * 8 * P + p * 64) * 16));
  };

  if constexpr (EPI == ROWPROJ_GELU)
    for (int i = tid; i < kGeluN; i += 256) gelu_t[i] = gelu_tail(__builtin_bit_cast(float, (kGeluLo + (uint32_t)i) << 16));

  // RMSNorm: 16 lanes per fp32 row (256-byte segments), LD rows in flight (all 32 where the registers hold them); the
  // bf16 rows pass, SL at a time, through the wave's part of the (still unused) ring into the fragment layout
  u32x4_t af[KS];
  {
    const int64_t rstride = is_s ? D : a.in_bstride;  // elements between the wave's rows
    constexpr int SL = D <= 384 ? 16 : 8, NV = D / 64, STR = 2 * D + 16;
    constexpr int LD = D <= 256 ? 32 : SL;  // rows in flight
    static_assert(4 * SL * STR <= NST * CHUNK, "the row scratch lies in the weight ring");
    char* sc = lds + wave * SL * STR;
    const float* x0 = a.x + (int64_t)b0 * a.in_bstride + (int64_t)t0 * D;
    const bool keep_h = EPI == ROWPROJ_GELU && part == 0 && a.h != nullptr;
    uint16_t* h0 = keep_h ? a.h + (int64_t)b0 * a.in_bstride + (int64_t)t0 * D : nullptr;
    const int sub = lane & 15, rq = lane >> 4;
    f32x4_t w[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) w[j] = *reinterpret_cast<const f32x4_t*>(a.norm_w + j * 64 + sub * 4);
    f32x4_t v[LD / 4][NV];
#pragma unroll
    for (int sl = 0; sl < 32 / SL; ++sl) {
      if (sl * SL % LD == 0) {
#pragma unroll
        for (int p = 0; p < LD / 4; ++p) {
          const float* xr = x0 + min(sl * SL + p * 4 + rq, last) * rstride + sub * 4;
#pragma unroll
          for (int j = 0; j < NV; ++j) v[p][j] = *reinterpret_cast<const f32x4_t*>(xr + j * 64);
        }
        // every load is in flight before the first is used (left to itself the compiler loads and reduces 4 rows at a
        // time, one memory latency each)
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int p = 0; p < SL / 4; ++p) {
        const f32x4_t(&u)[NV] = v[sl * SL % LD / 4 + p];
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j) ss += (u[j].x * u[j].x + u[j].y * u[j].y) + (u[j].z * u[j].z + u[j].w * u[j].w);
        ss = row16_sum(ss);
        const float rms = 1.0f / sqrtf(ss / (float)D + 1e-6f);
        const int r = sl * SL + p * 4 + rq;
        uint16_t* hr = h0 + (int64_t)r * rstride + sub * 4;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const u32x2_t n = u32x2_t{pack_bf16x2((u[j].x * rms) * w[j].x, (u[j].y * rms) * w[j].y),
                                    pack_bf16x2((u[j].z * rms) * w[j].z, (u[j].w * rms) * w[j].w)};
          if (keep_h && r < rows) *reinterpret_cast<u32x2_t*>(hr + j * 64) = n;
          *reinterpret_cast<u32x2_t*>(sc + (p * 4 + rq) * STR + j * 128 + sub * 8) = n;
        }
      }
      if (fr / SL == sl) {  // the wave's own LDS operations complete in order
#pragma unroll
        for (int s = 0; s < KS; ++s) af[s] = *reinterpret_cast<const u32x4_t*>(sc + (fr % SL) * STR + (2 * s + hf) * 16);
      }
    }
    __syncthreads();  // every wave is done with the scratch before the ring fills it
  }
#pragma unroll
  for (int j = 0; j < PF; ++j)
#pragma unroll
    for (int p = 0; p < NDMA; ++p) dma(min(c_begin + j, nchunks - 1), j, p);

  // Q is needed of the kept tail tokens only: rows below q_first of this wave have none
  const int q_first = a.kv - a.q_len - t0;
  const bool skip_q = EPI == ROWPROJ_QKV && (is_s ? q_first >= rows : rows == 0 || q_first > 0);

  // the previous chunk's tile, stored during the current one: line r (line_lo <= r < line_hi) at obase + r * ostride
  // elements, of which the first `outs` outputs exist
  f32x16_t prev;
#pragma unroll
  for (int e = 0; e < 16; ++e) prev[e] = 0.0f;
  uint16_t* obase = EPI == ROWPROJ_GELU ? a.out : a.k;
  uint32_t ostride = 0;
  int line_lo = 0, line_hi = 0, outs = 32;
  uint32_t pk[2][4];
  auto epi_pack = [&](int h) {
    if constexpr (EPI == ROWPROJ_GELU) {
      gelu2048_pack((uint32_t)(uintptr_t)lds + NST * CHUNK, prev, 8 * h, pk[h]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) pk[h][j] = pack_bf16x2(prev[8 * h + 2 * j], prev[8 * h + 2 * j + 1]);
    }
  };
  auto epi_store = [&](int i) {
    const int r = 16 * i + l16;
    const uint32_t off = ((uint32_t)r * ostride + piece * 8) * 2;
    store16(obase, r >= line_lo && r < line_hi && piece * 8 + 8 <= outs ? off : kNoStore,
            u32x4_t{pk[i][0], pk[i][1], pk[i][2], pk[i][3]});
  };
  // a sample's last V^T tokens when they are no multiple of 8: not the NS tokens behind them.  Four of them in one store
  // (blocks of 4,096 samples of 60 S and 4 NS tokens, d 128: 295 -> 288 us; any number of them in that way took more
  // registers and 303)
  auto epi_tail = [&]() {
    if (EPI == ROWPROJ_QKV && (outs & 7)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (piece == outs >> 3 && 16 * i + l16 < line_hi) {
          uint16_t* v = obase + (int64_t)(16 * i + l16) * ostride + piece * 8;
          if ((outs & 7) == 4) {
            *reinterpret_cast<u32x2_t*>(v) = u32x2_t{pk[i][0], pk[i][1]};
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (piece * 8 + e < outs) v[e] = (uint16_t)(pk[i][e >> 1] >> (16 * (e & 1)));
          }
        }
    }
  };

  int stg = 0;
  // chunk c: its MFMAs (V: columns on lanes; otherwise rows on lanes), then where its tile goes
  auto step = [&](int c, auto v_tag) {
    constexpr bool V = decltype(v_tag)::value;
    // Vector memory completes in issue order; behind chunk c's DMA the wave issued the DMAs of the PF - 1 chunks after
    // it and, from the PF-th chunk on, two stores in each of the PF iterations since: chunk c has landed once no more
    // than those are outstanding
    if (c - c_begin >= PF) __builtin_amdgcn_s_waitcnt(waitcnt_vm((PF - 1) * NDMA + PF * 2));
    else __builtin_amdgcn_s_waitcnt(waitcnt_vm((PF - 1) * NDMA));
    __syncthreads();  // publishes every wave's part of the chunk and frees the stage of chunk c - 1
    // past the end the last chunk is loaded again, into a stage that no later chunk reads
    const int cn = min(c + PF, nchunks - 1), sn = stg == 0 ? NST - 1 : stg - 1;
    // fragment s of the chunk: row fr, logical piece 2 s + hf, at slot (2 s) ^ (hf ^ (fr & 15)); rows and stages are
    // multiples of 256 bytes, so 8 XORed addresses and immediate offsets reach every fragment
    uint32_t wb = (uint32_t)(uintptr_t)lds + stg * CHUNK + fr * (2 * D) + ((hf ^ (fr & 15)) << 4);
    asm volatile("" : "+v"(wb));  // not hoisted out of the chunk loop: the variants would take 8 registers
    stg = stg + 1 == NST ? 0 : stg + 1;
    auto wfrag = [&](int s) {
      return reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(wb ^ ((2 * s & 15) << 4))[2 * s & ~15];
    };
    const bool is_q = EPI == ROWPROJ_QKV && !V && c * 32 < D;
    f32x16_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    if (is_q && skip_q) {
#pragma unroll
      for (int p = 0; p < NDMA; ++p) dma(cn, sn, p);
      epi_pack(0);
      epi_pack(1);
      tile_segments(pk);
      epi_store(0);
      epi_store(1);
    } else {
      // MFMAs of chunk c, with the DMAs and the previous chunk's epilogue between them (the order is pinned)
      u32x4_t wf[LEAD];
#pragma unroll
      for (int s = 0; s < LEAD; ++s) wf[s] = wfrag(s);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        acc = V ? mfma32x32x16(af[s], wf[s % LEAD], acc) : mfma32x32x16(wf[s % LEAD], af[s], acc);
        if (s + LEAD < KS) wf[s % LEAD] = wfrag(s + LEAD);
        if (s % 2 == 1 && s / 2 < NDMA) dma(cn, sn, s / 2);
        if (s == KS / 4) epi_pack(0);
        if (s == KS / 2) epi_pack(1);
        if (s == KS * 5 / 8) tile_segments(pk);
        if (s == KS * 6 / 8) epi_store(0);
        if (s == KS * 7 / 8) epi_store(1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    epi_tail();

    prev = acc;
    if constexpr (EPI == ROWPROJ_GELU) {
      obase = a.out + (int64_t)b0 * a.out_bstride + (int64_t)t0 * a.N + c * 32;
      ostride = is_s ? (uint32_t)a.N : (uint32_t)a.out_bstride;
      line_hi = rows;
    } else if constexpr (V) {
      // lines are features c*32 - 2D .. + 31, outputs the wave's tokens
      const int64_t vbs = (int64_t)D * a.kv_pad;  // elements per sample
      obase = a.vt + (int64_t)b0 * vbs + (int64_t)(c * 32 - 2 * D) * a.kv_pad + t0;
      ostride = (uint32_t)a.kv_pad;
      line_lo = 0;
      line_hi = is_s && rows > 0 ? 32 : 0;
      outs = is_s ? rows : 32;
      if (!is_s) {
        // one token of 32 samples: 2-byte stores at once, the sample stride added step by step
        int64_t vstep = vbs;
        asm volatile("" : "+s"(vstep));
        uint16_t* v = obase + (int64_t)(hf * 4) * vbs + (int64_t)fr * a.kv_pad;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          if ((e >> 2) * 8 + hf * 4 + (e & 3) < rows) *v = (uint16_t)bf16_bits(acc[e]);
          v += (e & 3) == 3 ? 5 * vstep : vstep;
        }
      }
    } else if (is_q) {
      obase = a.q + ((int64_t)b0 * a.q_len - q_first) * D + c * 32;
      ostride = is_s ? (uint32_t)D : (uint32_t)(a.q_len * D);
      line_lo = is_s ? max(q_first, 0) : 0;
      line_hi = skip_q ? 0 : rows;
    } else {
      obase = a.k + ((int64_t)b0 * a.kv + t0) * D + c * 32 - D;
      ostride = is_s ? (uint32_t)D : (uint32_t)(a.kv * D);
      line_lo = 0;
      line_hi = rows;
    }
  };
  int c = c_begin;
  const int c_v = EPI == ROWPROJ_QKV ? min(c_end, D / 16) : c_end;  // V chunks from 2 D columns on
  for (; c < c_v; ++c) step(c, std::false_type{});
  if constexpr (EPI == ROWPROJ_QKV)
    for (; c < c_end; ++c) step(c, std::true_type{});
  epi_pack(0);
  epi_pack(1);
  tile_segments(pk);
  epi_store(0);
  epi_store(1);
  epi_tail();
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // no DMA may land in LDS after the workgroup ends
}

template <int D, int EPI>
static int launch_one(RowProjArgs a, hipStream_t s) {
  constexpr int lds = rowproj_lds<D>(EPI == ROWPROJ_GELU);
  static std::once_flag once[64];
  static hipError_t err[64];
  int dev = 0;
  PDM_CHECK_HIP(hipGetDevice(&dev));
  PDM_CHECK_ARG(dev >= 0 && dev < 64, "device index out of range");
  std::call_once(once[dev], [&] {
    err[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(rowproj_kernel<D, EPI>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  });
  PDM_CHECK_HIP(err[dev]);
  // The S tokens behind a sample's last whole block: a block of their own, mostly padding when they are few, or tiles of
  // one token of 128 samples, like the NS tokens, without padding but with 2-byte V^T stores.  Tiles where they are few
  // enough workgroups: up to 16 tokens of many samples for the FFN-up, 6 for Q/K/V.  Whole blocks of 4,096 samples in
  // us, blocks / tiles for the FFN-up / tiles for both: d 512, 1 S token 769 / 561 / 464, 4 829 / 648 / 542, 8 925 / 788
  // / 768, 16 1,764 / 1,659 / 1,674, 28 1,453 / 1,430 / 1,504; Q/K/V alone (no NS tokens): d 128, 5 S tokens 73 / 71, 8
  // 70 / 82; d 384, 5 275 / 233, 8 312 / 303; d 256, 5 158 / 140, 8 155 / 163.
  const int tail = a.n_s % 32, whole = a.n_s - tail;
  a.tiles_b = (a.B + 127) / 128;
  auto blocks = [&](int n) { return ((int64_t)a.B * ((n + 31) / 32) + 3) / 4; };
  a.n_blk = (int64_t)tail * a.tiles_b * (EPI == ROWPROJ_QKV ? 5 : 2) <= blocks(a.n_s) - blocks(whole) ? whole : a.n_s;
  a.blocks_per_sample = (a.n_blk + 31) / 32;
  a.n_tok = a.n_s - a.n_blk + a.n_ns;
  const int64_t wgs_s = blocks(a.n_blk), wgs_tok = (int64_t)a.n_tok * a.tiles_b;
  // column splits: as many as keep the grid within one workgroup per CU, of at least two chunks each for the S tiles; a
  // second workgroup per CU only where the first round leaves no room for a split.  Every split reads and normalises its
  // tile's rows again, and at two per CU that took 5.0 us of a launch's 12 (one per CU 3.8; d 256, FFN-up of 16 samples
  // of 272 tokens).  One round against two, stacks in us: d 256 B = 16 198 / 202, B = 4 167 / 170, d 384 B = 8 810 / 830,
  // d 512 B = 4 305 / 321; without a split against two: d 256 B = 48 312 / 303, d 128 B = 100 194 / 183.
  // What is left of the round goes to the token tiles, down to single chunks: their weight is read from memory by few
  // workgroups, and their V^T goes out in 2-byte stores (500 samples of 98 tokens, d 384: Q/K/V 111 -> 81 us with the NS
  // tiles split).
  const int nchunks = a.N / 32;
  constexpr int64_t kCus = 256;
  const int64_t tiles = std::max<int64_t>(1, wgs_s + wgs_tok);
  const int64_t round = 2 * tiles <= kCus ? kCus : 2 * kCus;
  a.split_s = (int)std::max<int64_t>(1, std::min<int64_t>(nchunks / 2, round / tiles));
  a.split_tok = (int)std::max<int64_t>(1, std::min<int64_t>(nchunks, (round - wgs_s * a.split_s) / std::max<int64_t>(1, wgs_tok)));
  const int64_t grid = wgs_s * a.split_s + wgs_tok * a.split_tok;
  if (grid == 0) return PDM_OK;
  // a launch dimension holds less than 2^32 threads
  PDM_CHECK_ARG(grid < (int64_t(1) << 24), "row projection grid too large");
  // the 32 features of a V^T tile lie within 2^31 bytes of the first
  PDM_CHECK_ARG((int64_t)32 * a.kv_pad * 2 < (int64_t(1) << 31), "row projection rows too far apart");
  a.wgs_s = (int)wgs_s;
  a.wgs_tok = (int)wgs_tok;
  hipLaunchKernelGGL((rowproj_kernel<D, EPI>), dim3((unsigned)grid), dim3(256), lds, s, a);
  PDM_CHECK_LAUNCH();
  return PDM_OK;
}

template <int EPI>
static int launch_epi(const RowProjArgs& a, int D, hipStream_t s) {
  switch (D) {
    case 128: return launch_one<128, EPI>(a, s);
    case 256: return launch_one<256, EPI>(a, s);
    case 384: return launch_one<384, EPI>(a, s);
    case 512: return launch_one<512, EPI>(a, s);
    default: set_error("row projection: unsupported d_model"); return PDM_ERR_UNSUPPORTED;
  }
}

int launch_row_proj(const RowProjArgs& a, int D, int epi, hipStream_t s) {
  auto launch = [&](const RowProjArgs& r) {
    return epi == ROWPROJ_QKV ? launch_epi<ROWPROJ_QKV>(r, D, s) : launch_epi<ROWPROJ_GELU>(r, D, s);
  };
  // a wave's lines, the same token of up to 32 samples, lie within 2^31 bytes of its first: samples that are further
  // apart go out as many at a time as do
  const int64_t apart = 2 * (epi == ROWPROJ_QKV ? (int64_t)a.kv * D : a.out_bstride);
  const int64_t fit = std::max<int64_t>(1, ((int64_t(1) << 31) - 1) / apart);
  if (fit >= std::min(a.B, 32)) return launch(a);
  for (int64_t b = 0; b < a.B; b += fit) {
    RowProjArgs r = a;
    r.B = (int)std::min<int64_t>(fit, a.B - b);
    r.x += b * a.in_bstride;
    if (epi == ROWPROJ_QKV) {
      r.q += b * a.q_len * D;
      r.k += b * a.kv * D;
      r.vt += b * D * a.kv_pad;
    } else {
      if (r.h) r.h += b * a.in_bstride;
      r.out += b * a.out_bstride;
    }
    if (int st = launch(r)) return st;
  }
  return PDM_OK;
}

}  // namespace pdm
