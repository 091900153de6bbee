// NS tokens for gfx950: the NS input rows (scalar-feature rows and dense parts, bf16, zero-padded to a multiple of 64
// columns), then AutoSplitTokenizer's two Linear layers as tiled MFMA GEMMs with bias epilogues.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "pdm_common.h"
#include "mfma_common.h"

namespace pdm {

constexpr int kNsK = 64;  // column granularity of the GEMMs
// Samples from which a wave walks every part of its sample.  Whole calls in us, four waves per sample / one: 8 tables and 8
// dense parts (K 152, N 128) 1,024 samples 14.2 / 18.3, 4,096 20.1 / 21.2, 6,000 24.2 / 24.3, 30,000 74 / 69, 262,144 643 /
// 559; one dense part (K 513, N 128) 15.3 / 15.4, 20.3 / 19.4,
// 25.0 / 22.4, 56 / 44, 551 / 405; the 4 + 4 parts of K 396, N 256 15.3 / 17.4, 23.1 / 23.8, 28.5 / 28.2, 77 / 70, 676 / 600.
constexpr int64_t kNsSplitSamples = 5000;

struct NsArgs {
  const char* tables[PDM_NS_MAX_PARTS];
  const int64_t* ids[PDM_NS_MAX_PARTS];
  int64_t rows[PDM_NS_MAX_PARTS];
  const float* dense[PDM_NS_MAX_PARTS];
  int64_t dense_stride[PDM_NS_MAX_PARTS];
  int32_t col[2 * PDM_NS_MAX_PARTS + 1];  // first column of part j (scalar parts, then dense parts)
  int32_t n_scalar, n_parts, f32_tables, K, K64;
  int64_t B;
  uint16_t* raw;  // [B, K64] bf16
  const uint16_t* w1;  // [N, K]
  uint16_t* w1p;       // [N, K64]
  int32_t N;
  int64_t w1p_elems;  // 0: W1 is read where it is
  int64_t row_blocks;  // blocks that write rows of raw
  int32_t split;       // waves per sample: 4 or 1
  int32_t* err;
};

// Rows of raw and the columns that pad W1, in one launch.  The first row_blocks blocks: a sample per `split` waves, which
// share out its parts, lanes over a part's columns, bf16 (round to nearest even) out.  The blocks after them: W1 [N, K] ->
// [N, K64] with zero columns K .. K64, 4 columns a thread.  Four waves per sample while the samples leave the card room:
// the parts' id -> row chains run beside each other (1,024 samples of 8 parts: a wave per sample walking every part took
// 8 us, W1's padding in a launch of its own another 5; together 5 us).
__global__ __launch_bounds__(256) void ns_prep_kernel(NsArgs a) {
  const int64_t block = linear_block();
  if (block >= a.row_blocks) {
    const int64_t i = ((block - a.row_blocks) * 256 + threadIdx.x) * 4;
    if (i >= a.w1p_elems) return;
    const int n = (int)(i / a.K64), k = (int)(i - (int64_t)n * a.K64);
    const uint16_t* src = a.w1 + (int64_t)n * a.K;
    uint32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = src[min(k + e, a.K - 1)];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < a.K ? v[e] : 0u;
    *reinterpret_cast<u32x2_t*>(a.w1p + i) = u32x2_t{v[0] | v[1] << 16, v[2] | v[3] << 16};
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t b = a.split == 4 ? block : block * 4 + wave;
  const int part0 = a.split == 4 ? wave : 0;
  if (b >= a.B) return;
  uint16_t* dst = a.raw + b * a.K64;
  bool bad = false;
  for (int j = part0; j < a.n_parts; j += a.split) {
    const int c0 = a.col[j], w = a.col[j + 1] - c0;
    if (j < a.n_scalar) {
      const int64_t id = a.ids[j][b];
      const bool ok = id >= 0 && id < a.rows[j];
      bad |= !ok;
      if (!ok) {
        for (int c = lane; c < w; c += 64) dst[c0 + c] = 0;
      } else if (a.f32_tables) {
        const float* row = reinterpret_cast<const float*>(a.tables[j]) + id * w;
        for (int c = lane; c < w; c += 64) dst[c0 + c] = (uint16_t)f32_to_bf16_bits(row[c]);
      } else {
        const uint16_t* row = reinterpret_cast<const uint16_t*>(a.tables[j]) + id * w;
        for (int c = lane; c < w; c += 64) dst[c0 + c] = row[c];
      }
    } else {
      const int d = j - a.n_scalar;
      const float* row = a.dense[d] + b * a.dense_stride[d];
      for (int c = lane; c < w; c += 64) dst[c0 + c] = (uint16_t)f32_to_bf16_bits(row[c]);
    }
  }
  if (part0 == a.split - 1)
    for (int c = a.K + lane; c < a.K64; c += 64) dst[c] = 0;
  if (bad && a.err) a.err[0] = 1;
}

// The tokenizer's Linear layers: out = epilogue(A . W^T + bias), A [M, K] rows with stride a_stride, W [N, K].
enum { NS_BIAS_GELU = 0, NS_BIAS_F32 = 1 };
struct NsGemmArgs {
  const uint16_t* A;
  int64_t a_stride;
  const uint16_t* W;
  const uint16_t* bias;  // bf16 [N]
  int M, N, K;           // K a multiple of 64, N of 64
  void* out;             // bf16 (NS_BIAS_GELU) or fp32 (NS_BIAS_F32) rows, stride out_stride
  int64_t out_stride;
  int tiles_m, tiles_n;
};

// four floats at any float's address (the caller's rows need no 16-byte alignment)
typedef float f32x4_a4_t __attribute__((ext_vector_type(4), aligned(4)));

// Tiles of TM rows x TN columns, eight waves: WM x WN wave tiles, each computed by KW waves that share out the k slabs
// (16 columns) of a stage, so that every SIMD has two waves to issue.  A and W stream global -> LDS by LDS DMA into a
// ring of NST stages of BK columns, NST ahead.  The fragments of stage kt + 1 are read into registers between the MFMAs
// of stage kt: a stage's slot is free as soon as its fragments are read, and the LDS reads (as long as the MFMAs at
// 128 x 128) no longer wait in front of them behind the barrier.  A row of a stage holds 16-byte piece v at slot
// v ^ swz(row), which spreads the rows of a fragment read over the banks.  Rows past M or N read the last row and are
// not stored.
//
// What bounds it, 1,024 rows, N = K = 4,096 (34 GFLOP, 14 us of MFMA at 128 x 128 on 256 CUs; 42 MB, 9 us): per stage
// and CU 512 cycles of MFMA, 512 of LDS reads, 256 of LDS writes by the DMA and as much again of the L2's 64 bytes per
// cycle.  With the reads behind the barrier these added up: Linear 2 48 us, Linear 1 (K = 396) 22 us, of which most was
// an epilogue of 2-byte stores by half of the waves; now 37 and 13 us.
//
// Epilogue: wave tiles are cut into 32-row blocks, each finished by one of the tile's KW waves: the others leave their
// sums in LDS, the finisher adds them in wave order and passes the block through LDS again, so that the stores take
// whole row segments.
template <int EPI, int TM, int TN, int WM, int WN, int BK, int NST>
__global__ __launch_bounds__(512, 1) void ns_gemm_kernel(NsGemmArgs a) {
  constexpr int KW = 8 / (WM * WN), MB = TM / WM / 32, NB = TN / WN / 32;
  constexpr int S = BK / 16 / KW;              // k slabs per wave and stage
  constexpr int RB = BK * 2, LPR = BK / 8;     // bytes and 16-byte pieces per row of a stage
  constexpr int STAGE = (TM + TN) * RB, NDMA = STAGE / 8192;  // DMA instructions per wave and stage
  static_assert(S >= 1 && NDMA * 8192 == STAGE && TM * RB % 1024 == 0, "a stage splits evenly over the waves");
  constexpr int SROW = NB * 128 + 16;          // LDS bytes per staged output row
  static_assert(KW >= 2 && WM * WN * MB * (KW - 1) * 32 * SROW <= NST * STAGE, "the sums must fit in the ring");
  extern __shared__ __attribute__((aligned(256))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int q = wave % (WM * WN), kw = wave / (WM * WN), wm = q / WN, wn = q % WN;
  int mt, nt;
  {
    const int bid = (int)blockIdx.x;
    if (a.tiles_n % 8 == 0) {  // XCD x (workgroups go to the 8 in turn) takes an eighth of the columns, all rows
      const int j = bid >> 3;
      mt = j % a.tiles_m;
      nt = (bid & 7) * (a.tiles_n / 8) + j / a.tiles_m;
    } else {
      mt = bid / a.tiles_n;
      nt = bid - mt * a.tiles_n;
    }
  }
  const int m0 = mt * TM, n0 = nt * TN;

  auto swz = [](int r) { return BK == 64 ? (r >> 1) & 7 : r & 15; };
  // instruction p of a wave fills 64 / LPR rows of the stage (A's rows, then W's)
  uint32_t off[NDMA];
  uint64_t base[NDMA];
#pragma unroll
  for (int p = 0; p < NDMA; ++p) {
    const int r0 = (wave * NDMA + p) * (64 / LPR);
    const bool is_a = r0 < TM;  // wave-uniform: TM is a multiple of 64 / LPR
    const int r = r0 - (is_a ? 0 : TM) + lane / LPR;
    const int row = is_a ? min(m0 + r, a.M - 1) - m0 : min(n0 + r, a.N - 1) - n0;
    off[p] = (uint32_t)(((int64_t)row * (is_a ? a.a_stride : (int64_t)a.K) + ((lane % LPR) ^ swz(r)) * 8) * 2);
    base[p] = (uint64_t)(uintptr_t)(is_a ? a.A + (int64_t)m0 * a.a_stride : a.W + (int64_t)n0 * a.K);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  auto dma = [&](int kt, int stg) {
#pragma unroll
    for (int p = 0; p < NDMA; ++p)
      lds_dma16(base[p] + (uint64_t)kt * RB, off[p], lds0 + stg * STAGE + (wave * NDMA + p) * 1024);
  };

  f32x16_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // fragment (row block, slab s of this wave): row fr, piece 2 (kw S + s) + hf
  const uint32_t ra = (uint32_t)((wm * MB * 32 + fr) * RB), rw = (uint32_t)((TM + wn * NB * 32 + fr) * RB);
  uint32_t po[S];
#pragma unroll
  for (int s = 0; s < S; ++s) po[s] = (uint32_t)(((2 * (kw * S + s) + hf) ^ swz(fr)) << 4);
  u32x4_t af[2][S][MB], wf[2][S][NB];
  auto fread = [&](int stg, int s, u32x4_t (&fa)[MB], u32x4_t (&fw)[NB]) {
    const uint32_t sb = lds0 + stg * STAGE + po[s];
#pragma unroll
    for (int i = 0; i < MB; ++i)
      fa[i] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(sb + ra + i * 32 * RB);
#pragma unroll
    for (int j = 0; j < NB; ++j)
      fw[j] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(sb + rw + j * 32 * RB);
  };

  const int nk = a.K / BK;
#pragma unroll
  for (int j = 0; j < NST; ++j) dma(min(j, nk - 1), j);
  // DMAs complete in issue order: stage 0 has landed once only the NST - 1 after it are outstanding
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((NST - 1) * NDMA));
  __syncthreads();
#pragma unroll
  for (int s = 0; s < S; ++s) fread(0, s, af[0][s], wf[0][s]);
  int stg = 0;
  // stage kt is in the fragments of set CUR; reads stage kt + 1 into the other
  auto step = [&](int kt, auto cur_tag) {
    constexpr int CUR = decltype(cur_tag)::value;
    // of the stages issued (.. kt + NST - 1) those after kt + 1 may still be outstanding
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((NST - 2) * NDMA));
    __syncthreads();  // publishes stage kt + 1; every wave has read its fragments of stage kt, whose slot is free
    dma(min(kt + NST, nk - 1), stg);  // past the end: the last one again, read by nobody
    stg = stg + 1 == NST ? 0 : stg + 1;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      fread(stg, s, af[CUR ^ 1][s], wf[CUR ^ 1][s]);  // after the last stage: an old one, used by nobody
      // rows on lanes: acc[i][j] holds row i*32 + fr, columns j*32 + (e/4)*8 + hf*4 + e%4
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma32x32x16(wf[CUR][s][j], af[CUR][s][i], acc[i][j]);
    }
  };
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    step(kt, std::integral_constant<int, 0>{});
    step(kt + 1, std::integral_constant<int, 1>{});
  }
  if (kt < nk) step(kt, std::integral_constant<int, 0>{});
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // no DMA may land in LDS once the epilogue uses it
  __syncthreads();

  // block i of wave tile q is finished by wave kw = i % KW; slot (q, i, the kw-th of the others)
  auto slot = [&](int i, int k) { return lds + ((q * MB + i) * (KW - 1) + k) * 32 * SROW; };
  auto piece = [&](char* st, int j, int g) { return reinterpret_cast<f32x4_t*>(st + fr * SROW + j * 128 + g * 32 + hf * 16); };
#pragma unroll
  for (int i = 0; i < MB; ++i)
    if (i % KW != kw) {
      char* st = slot(i, kw < i % KW ? kw : kw - 1);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *piece(st, j, g) = f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    }
  __syncthreads();
  constexpr int LR = NB * 8, RPI = 64 / LR;  // lanes per row, rows per store instruction
  const int col = n0 + wn * NB * 32 + (lane % LR) * 4;
#pragma unroll
  for (int i = 0; i < MB; ++i)
    if (i % KW == kw) {
      char* st = slot(i, 0);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4_t v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
#pragma unroll
          for (int k = 0; k < KW - 1; ++k) {
            const f32x4_t o = *piece(slot(i, k), j, g);
            v = f32x4_t{v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w};
          }
          *piece(st, j, g) = v;  // the wave's own LDS operations complete in order
        }
      if (col < a.N) {
        float bias[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[e] = bf16_bits_to_f32(a.bias[col + e]);
#pragma unroll
        for (int r = 0; r < 32; r += RPI) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(st + (r + lane / LR) * SROW + (lane % LR) * 16);
          const int m = m0 + (wm * MB + i) * 32 + r + lane / LR;
          if (m >= a.M) continue;
          // one rounding after the bias, as autocast makes it; then the GELU in bf16, or the bf16 result as fp32
          const float x[4] = {bf16_round(v.x + bias[0]), bf16_round(v.y + bias[1]), bf16_round(v.z + bias[2]), bf16_round(v.w + bias[3])};
          if constexpr (EPI == NS_BIAS_GELU)
            *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)m * a.out_stride + col) =
                u32x2_t{pack_bf16x2(gelu_erf(x[0]), gelu_erf(x[1])), pack_bf16x2(gelu_erf(x[2]), gelu_erf(x[3]))};
          else
            *reinterpret_cast<f32x4_a4_t*>(reinterpret_cast<float*>(a.out) + (int64_t)m * a.out_stride + col) =
                f32x4_a4_t{x[0], x[1], x[2], x[3]};
        }
      }
    }
}

template <int EPI, int TM, int TN, int WM, int WN, int BK, int NST>
static int launch_ns_tiles(NsGemmArgs a, hipStream_t s) {
  a.tiles_m = (a.M + TM - 1) / TM;
  a.tiles_n = (a.N + TN - 1) / TN;
  const int64_t grid = (int64_t)a.tiles_m * a.tiles_n;
  PDM_CHECK_ARG(grid < (int64_t(1) << 31), "GEMM grid too large");
  // 32-bit per-lane DMA offsets within a tile's rows
  PDM_CHECK_ARG((int64_t)128 * std::max<int64_t>(a.a_stride, a.K) * 2 < (int64_t(1) << 31), "rows too long");
  constexpr int bytes = NST * (TM + TN) * BK * 2;
  static std::once_flag once[64];
  static hipError_t err[64];
  int dev = 0;
  PDM_CHECK_HIP(hipGetDevice(&dev));
  PDM_CHECK_ARG(dev >= 0 && dev < 64, "device index out of range");
  const auto kernel = ns_gemm_kernel<EPI, TM, TN, WM, WN, BK, NST>;
  std::call_once(once[dev], [&] {
    err[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  });
  PDM_CHECK_HIP(err[dev]);
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), bytes, s, a);
  PDM_CHECK_LAUNCH();
  return PDM_OK;
}

template <int EPI>
static int launch_ns_gemm(const NsGemmArgs& a, hipStream_t s) {
  // 64 x 64 tiles while one round of them (one per CU) holds the output: twice the tiles of either side in flight, a
  // four-way split of k.  Linear 2 of 4,096 outputs, both sides in us (64 against 128): 16 rows 14.4 / 25.4, 128 rows
  // 15.4 / 27.3, 256 rows (one full round) 17.0 / 27.3, 384 rows 29.6 / 28.2, 1,024 rows 75 / 37.
  const int64_t tiles = (int64_t)((a.M + 63) / 64) * ((a.N + 63) / 64);
  if (tiles <= 256) return launch_ns_tiles<EPI, 64, 64, 2, 1, 64, 8>(a, s);
  return launch_ns_tiles<EPI, 128, 128, 2, 2, 64, 4>(a, s);
}

static int64_t align256(int64_t v) { return (v + 255) & ~int64_t(255); }

struct NsLayout {
  int64_t raw, h, w1p, total;
};

// Row stride (elements) of the hidden activations h: N plus one 128-byte line, so that the rows an XCD's
// tiles read at one k step do not all fall into the same few L2 sets (N is a multiple of 64).
static int64_t ns_h_stride(int64_t N) { return N + 64; }

static NsLayout ns_layout(int64_t B, int64_t K64, int64_t N) {
  NsLayout l{};
  l.raw = 0;
  l.h = align256(B * K64 * 2);
  l.w1p = l.h + align256(B * ns_h_stride(N) * 2);
  l.total = l.w1p + align256(N * K64 * 2);
  return l;
}

static const char* check_ns_desc(const pdm_ns_desc* d, int& K) {
  if (!d) return "null desc";
  if (d->num_scalar < 0 || d->num_scalar > PDM_NS_MAX_PARTS || d->num_dense < 0 || d->num_dense > PDM_NS_MAX_PARTS)
    return "num_scalar and num_dense must be in [0, 8]";
  if (d->num_scalar + d->num_dense == 0) return "no NS input parts";
  if (d->table_dtype != PDM_F32 && d->table_dtype != PDM_BF16) return "table_dtype must be F32 or BF16";
  if (d->n_out < 8 || d->n_out % 8 != 0) return "n_out must be a positive multiple of 8";
  if (d->batch_size < 0) return "batch_size < 0";
  K = 0;
  for (int j = 0; j < d->num_scalar; ++j) {
    if (d->scalar_dim[j] <= 0 || d->scalar_rows[j] < 0) return "bad scalar table shape";
    K += d->scalar_dim[j];
  }
  for (int j = 0; j < d->num_dense; ++j) {
    if (d->dense_dim[j] <= 0) return "bad dense part width";
    K += d->dense_dim[j];
  }
  return nullptr;
}

}  // namespace pdm

using namespace pdm;

extern "C" int64_t pdm_ns_tokenize_workspace_size(const pdm_ns_desc* desc) {
  clear_error();
  int K = 0;
  if (const char* e = check_ns_desc(desc, K)) {
    set_error(std::string("pdm_ns_tokenize_workspace_size: ") + e);
    return -1;
  }
  return ns_layout(desc->batch_size, (K + kNsK - 1) / kNsK * kNsK, desc->n_out).total;
}

extern "C" int pdm_ns_tokenize_fwd(const pdm_ns_desc* desc, const void* const* tables, const int64_t* const* ids,
                                   const float* const* dense, const int64_t* dense_stride, const uint16_t* w1,
                                   const uint16_t* b1, const uint16_t* w2, const uint16_t* b2, float* out,
                                   int64_t out_sample_stride, void* workspace, int64_t workspace_bytes,
                                   int32_t* err_flag, pdm_stream_t stream) {
  clear_error();
  int K = 0;
  if (const char* e = check_ns_desc(desc, K)) {
    set_error(std::string("pdm_ns_tokenize_fwd: ") + e);
    return PDM_ERR_INVALID;
  }
  const pdm_ns_desc& d = *desc;
  const int N = d.n_out;
  const int K64 = (K + kNsK - 1) / kNsK * kNsK;
  if (d.batch_size == 0) return PDM_OK;
  PDM_CHECK_ARG(d.batch_size < (int64_t(1) << 31), "batch_size too large");
  PDM_CHECK_ARG(w1 && b1 && w2 && b2 && out, "null weight or output pointer");
  PDM_CHECK_ARG(((uintptr_t)w2 & 15) == 0 && ((uintptr_t)w1 & 1) == 0, "w2 must be 16-byte aligned");
  PDM_CHECK_ARG(out_sample_stride >= N, "out_sample_stride must be >= n_out");
  PDM_CHECK_ARG(N % kNsK == 0, "n_out must be a multiple of 64");
  NsArgs a{};
  a.n_scalar = d.num_scalar;
  a.n_parts = d.num_scalar + d.num_dense;
  a.f32_tables = d.table_dtype == PDM_F32;
  int col = 0;
  for (int j = 0; j < d.num_scalar; ++j) {
    PDM_CHECK_ARG(tables && ids && tables[j] && ids[j], "null scalar table or ids pointer");
    a.tables[j] = reinterpret_cast<const char*>(tables[j]);
    a.ids[j] = ids[j];
    a.rows[j] = d.scalar_rows[j];
    a.col[j] = col;
    col += d.scalar_dim[j];
  }
  for (int j = 0; j < d.num_dense; ++j) {
    PDM_CHECK_ARG(dense && dense_stride && dense[j], "null dense pointer");
    PDM_CHECK_ARG(dense_stride[j] >= d.dense_dim[j], "dense_stride must be >= dense_dim");
    a.dense[j] = dense[j];
    a.dense_stride[j] = dense_stride[j];
    a.col[d.num_scalar + j] = col;
    col += d.dense_dim[j];
  }
  a.col[a.n_parts] = col;
  a.K = K;
  a.K64 = K64;
  a.B = d.batch_size;
  a.err = err_flag;
  const NsLayout lay = ns_layout(d.batch_size, K64, N);
  PDM_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
  PDM_CHECK_ARG(workspace_bytes >= lay.total, "workspace too small");
  char* ws = reinterpret_cast<char*>(workspace);
  a.raw = reinterpret_cast<uint16_t*>(ws + lay.raw);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + lay.h);
  uint16_t* w1p = reinterpret_cast<uint16_t*>(ws + lay.w1p);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);

  // W1 with rows of whole 64-column stages, 16-byte aligned, is read where it is
  const bool pad = K != K64 || ((uintptr_t)w1 & 15) != 0;
  a.w1 = w1;
  a.w1p = w1p;
  a.N = N;
  a.w1p_elems = pad ? (int64_t)N * K64 : 0;
  a.split = d.batch_size < kNsSplitSamples ? 4 : 1;
  a.row_blocks = a.split == 4 ? d.batch_size : (d.batch_size + 3) / 4;
  hipLaunchKernelGGL(ns_prep_kernel, linear_grid(a.row_blocks + (a.w1p_elems / 4 + 255) / 256), dim3(256), 0, s, a);
  PDM_CHECK_LAUNCH();
  NsGemmArgs g{};
  g.M = (int)d.batch_size;
  g.N = N;
  // Linear 1: h = bf16(gelu(bf16(raw . W1^T + b1)))
  g.A = a.raw;
  g.a_stride = K64;
  g.W = pad ? w1p : w1;
  g.K = K64;
  g.bias = b1;
  g.out = h;
  g.out_stride = ns_h_stride(N);
  if (int st = launch_ns_gemm<NS_BIAS_GELU>(g, s)) return st;
  // Linear 2: out = float(bf16(h . W2^T + b2))
  g.A = h;
  g.a_stride = ns_h_stride(N);
  g.W = w2;
  g.K = N;
  g.bias = b2;
  g.out = out;
  g.out_stride = out_sample_stride;
  return launch_ns_gemm<NS_BIAS_F32>(g, s);
}
