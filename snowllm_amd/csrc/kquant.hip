// GGUF Q4_K / Q8_0 dequant-GEMV for short verify blocks (M <= 16 rows per pass) on gfx950:
// repack, activation prep and the plain GEMV (shared device code in kquant_core.h).
//
// Weights stay packed in HBM. A one-time repack (snowllm_gemm_kquant_shuffle_b) moves the
// GGUF bytes into MFMA lane order: a 16-column tile of one 256-weight superblock is a single
// contiguous 2 KiB run of nibbles (Q4_K) or 4 KiB of int8 (Q8_0), read with 16-byte loads
// that are fully coalesced across the wave, plus 16 bytes of block header per column.
//
// Arithmetic (per 32-weight sub-block j, column n, row r):
//   y[r,n] = sum_j  a_j * sum_i q_i x_ri  - mn_j * sum_i x_ri
// Quants are turned into exact fp16 values with the 1024-offset trick (0x6400 | q == 1024+q;
// a high nibble left in bits 4..7 reads as 1024+16q), multiplied against fp16 activations on
// v_mfma_f32_16x16x32_f16 (K = 32 = one sub-block), and the sub-block result is scaled by
// a_j in fp32. The offset and min terms are one rank-8 product per superblock, done on
// v_mfma_f32_16x16x4_f32 with the sub-block sums of the activations. Activations are
// converted to fp16 once per call with a power-of-two scale per (row, superblock), exact for
// bf16 input.
#include "kquant_core.h"

#include <mutex>
#include <type_traits>

namespace {
using namespace kq;

// ---------------------------------------------------------------------------------------
// Activation prep kernel: one wave per (row tile, superblock), writing the workspace.
// ---------------------------------------------------------------------------------------
__global__ void __launch_bounds__(64) xprep_kernel(const uint16_t* __restrict__ a, int64_t M,
                                                   int64_t K, void* ws, size_t tile_bytes) {
  const int s = blockIdx.x, tile = blockIdx.y;
  const int lane = threadIdx.x;
  const int64_t S = K / QK;
  XPrepView v = xprep_view((char*)ws + tile * tile_bytes, S);
  const int64_t r0 = (int64_t)tile * TILE_M;
  XOperands o;
  convert_superblock(a + r0 * K, K, (int)(M - r0 < TILE_M ? M - r0 : TILE_M), s, lane, o);
  store_operands(v, s, lane, o);
}

// NW waves split the superblocks of NTILE column tiles; the waves' partial sums meet in LDS
// and are added in a fixed order. A last partial tile group reads its last tile again and
// writes it once.
// RAW: ws is the bf16 activation matrix [M, S*256] itself, converted in-kernel (one launch
// for the whole operator instead of a prep pass + GEMV).
template <int FMT, int NTILE, int NW, bool RAW = false>
__global__ void __launch_bounds__(NW * 64) kquant_gemv(const u32x4* __restrict__ quant,
                                                       const u32x4* __restrict__ meta,
                                                       const void* __restrict__ ws,
                                                       void* __restrict__ c, int M, int N, int S,
                                                       int c_bf16, int ldc) {
  __shared__ floatx4 part[NW][NTILE][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int kq = lane >> 4;
  const int tiles = N / TILE_N;
  const int tile0 = blockIdx.x * NTILE;
  GemvStreams st = make_streams<FMT>(quant, meta, ws, tiles, S, lane, M);
  if constexpr (NTILE > 1) st.last = tiles - 1;
  const uint32_t Mv = decode_magic<FMT>();
  floatx4 acc[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (RAW) {
    const RawX rx = make_raw_x(ws, M, S * QK, lane);
    gemv_loop_raw<FMT, NTILE, NW>(st, rx, w, S, tile0, 1, lane, Mv, acc);
  } else {
    gemv_loop<FMT, NTILE, NW>(st, w, S, tile0, 1, kq, Mv, acc);
  }
  combine_waves<NTILE, NW>(part, acc, w, lane);
  for (int idx = threadIdx.x; idx < NTILE * 64; idx += NW * 64) {
    const int t = idx >> 6, l = idx & 63;
    const int tile = tile0 + t;
    if (tile >= tiles) continue;
    floatx4 v = part[0][t][l];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) v += part[ww][t][l];
    const int n = tile * TILE_N + (l & 15);
    const int rb = 4 * (l >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = rb + i;
      if (row >= M) break;
      if (c_bf16) ((uint16_t*)c)[(int64_t)row * ldc + n] = f32_to_bf16(v[i]);
      else ((float*)c)[(int64_t)row * ldc + n] = v[i];
    }
  }
}

// ---------------------------------------------------------------------------------------
// The same GEMV over MT 16-row tiles at once (a verify step wider than 16 rows; blockIdx.y: the
// group of MT tiles): each wave decodes a superblock of NT column tiles once for the prepared
// operands of MT row tiles (gemv_rows_loop). Bound: the L2 reads (26 KB per 2 x 4 tiles and
// superblock, 13 KB per 1 x 2) and the vector units' decode and rescaling, both shared by more
// tiles the more a wave holds: Q4_K 2 x 4, 4096 x 14336, 126 rows, reads 388 MB from L2 in 33 us
// (11.8 TB/s) with the vector units 48 % busy; Q6_K 1 x 2, 151,936 x 2048, 45 rows, 1.72 GB in
// 150 us (11.4 TB/s) and 72 %, its weights fetched into L2 once per row tile (767 MB). Two row tiles take the registers of two waves per SIMD, one
// workgroup to a CU; one row tile is held to four waves per SIMD, two workgroups (above 128
// registers Q8_0 took 10 to 15 % longer, 17.8 us against 15.3 at 5120 x 2048 and 128 rows). Q4_K
// 4096 x 14336, 126 rows, with the operands' launch: 47 -> 38 us from HBM, 42 -> 32 repeated,
// against one row tile by two column tiles with no load ahead.
// The per-row arithmetic and the waves' superblock split are those of kquant_gemv with NW waves, so
// every row gets the bits of the 16-row launch.
// ---------------------------------------------------------------------------------------
template <int FMT, int NW, int MT, int NT>
__global__ void __launch_bounds__(NW * 64)
    __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2))) kquant_gemv_mt(const u32x4* __restrict__ quant,
                                                          const u32x4* __restrict__ meta,
                                                          const void* __restrict__ ws,
                                                          void* __restrict__ c, int M, int N,
                                                          int S, int c_bf16, size_t tile_bytes,
                                                          int ldc) {
  __shared__ floatx4 part[NW][NT][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = N / TILE_N;
  const int tile0 = blockIdx.x * NT;  // NT column tiles share each row tile's operands
  const int m0 = blockIdx.y * MT;
  const int row_tiles = (M + TILE_M - 1) / TILE_M;
  GemvStreams st = make_streams<FMT>(quant, meta, ws, tiles, S, lane, 16);
  if constexpr (NT > 1) st.last = tiles - 1;
  const uint32_t Mv = decode_magic<FMT>();
  floatx4 acc[MT][NT];
  // (one row tile of Q8_0 has no registers for the next superblock at four waves per SIMD)
  constexpr bool AHEAD = !(FMT == FMT_Q8_0 && MT == 1);
  gemv_rows_loop<FMT, MT, NT, NW, AHEAD>(st, ws, tile_bytes, M, m0, S, lane, w,
                                         [&](int t) { return tile0 + t; }, Mv, acc);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m0 + m >= row_tiles) break;  // uniform
    if (m) __syncthreads();
    combine_waves<NT, NW>(part, acc[m], w, lane);
    for (int idx = threadIdx.x; idx < NT * 64; idx += NW * 64) {
      const int t = idx >> 6, l = idx & 63;
      const int tile = tile0 + t;
      if (tile >= tiles) continue;
      floatx4 v = part[0][t][l];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) v += part[ww][t][l];
      const int n = tile * TILE_N + (l & 15);
      const int rb = (m0 + m) * TILE_M + 4 * (l >> 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = rb + i;
        if (row >= M) break;
        if (c_bf16) ((uint16_t*)c)[(int64_t)row * ldc + n] = f32_to_bf16(v[i]);
        else ((float*)c)[(int64_t)row * ldc + n] = v[i];
      }
    }
  }
}

template <int FMT, int NW>
int launch_gemv_mt(const void* quant, const void* meta, const void* ws, void* c, int M, int N,
                   int S, int c_bf16, int ldc, hipStream_t s) {
  const int tiles = N / TILE_N;
  const int row_tiles = (M + TILE_M - 1) / TILE_M;
  const size_t tb = xprep_tile_bytes(S);
  auto go = [&](auto kern, int mt, int ntile) {
    hipLaunchKernelGGL(kern, dim3((tiles + ntile - 1) / ntile, (row_tiles + mt - 1) / mt),
                       dim3(NW * 64), 0, s, (const u32x4*)quant, (const u32x4*)meta, ws, c, M,
                       N, S, c_bf16, tb, ldc);
  };
  // One row tile per workgroup, by two column tiles where that leaves 192 or more workgroups (two
  // of them to a CU), or two row tiles by four or two column tiles (one workgroup to a CU): the form
  // of the least estimated time. In units of 1024 tile products, one round of the 256 CUs for
  // 1 x 2 and 2 x 2 and half a round for 2 x 4, the estimate is the form's rounds over its speed
  // against 1 x 2 when full. Two-row workgroups run in whole rounds; the smaller ones' last round
  // is partly hidden. An odd last row tile costs a two-row form a whole one. The speeds and the
  // rule are fitted to 450 sizes a format (18 N x K from 512 x 2048 to 151,936 x 2048, 17 to 256
  // rows; MI355X, operands' launch included, weights from HBM): on average 1.0 to 1.4 % above each
  // size's best form. Against one row tile without a load ahead 7 % (Q4_K), 4 % (Q5_K), 29 % (Q6_K)
  // and 14 % (Q8_0) faster on average and slower nowhere, but for up to 0.4 us of 11 at 4 sizes of
  // Q8_0; a rule on the last round's fill alone lost to it by up to 15 %. us, 1 x 2 / 2 x 2 / 2 x 4:
  //   4096 x 14336, 126 rows   Q4_K 46 / 43 / 38      Q6_K 63 / 51 / 47
  //   14336 x 4096, 108 rows   Q4_K 43 / 48 / 45      Q5_K 56 / 59 / -
  //   8192 x 8192, 256 rows    Q5_K 133 / 114 / -
  //   28672 x 4096, 240 rows   Q8_0 257 / 216 / 181
  //   5120 x 2048, 128 rows    Q8_0 15.3 / 18.5 / 17.4
  //   151936 x 2048, 45 rows   Q6_K 144 / 175 / 155   Q4_K 121 / 147 / 126   Q8_0 199 / 210 / 172
  // Below eight superblocks two-row forms would leave half their waves idle. Q5_K's 2 x 4 spills
  // and its 2 x 2 needs two superblocks per wave (K = 2048 at 240 rows: 1.16 times as long); Q4_K's
  // and Q8_0's 2 x 2 is behind 1 x 2 or 2 x 4 everywhere.
  const bool two = (int64_t)(tiles / 2) * row_tiles >= 192;
  if constexpr (NW == 8) {
    const double w24 = FMT == FMT_Q4_K ? 1.1 : 1.3, w22 = FMT == FMT_Q5_K ? 1.02 : 1.1;
    const int64_t pairs = (row_tiles + 1) / 2;
    auto rounds = [&](int ntile) { return (double)(((tiles + ntile - 1) / ntile * pairs + 255) / 256); };
    const int64_t small = two ? (tiles + 1) / 2 * (int64_t)row_tiles : (int64_t)tiles * row_tiles;
    const double x = (double)small / 512, t1 = (x + (double)((small + 511) / 512)) / (two ? 2 : 4);
    const double t24 = 2 * rounds(4) / w24, t22 = rounds(2) / w22;
    if constexpr (FMT != FMT_Q5_K) {
      if (t24 < t1 && (FMT != FMT_Q6_K || t24 <= t22)) {
        go(kquant_gemv_mt<FMT, NW, 2, 4>, 2, 4);
        SV_CHECK_LAUNCH();
        return SV_OK;
      }
    }
    if constexpr (FMT == FMT_Q5_K || FMT == FMT_Q6_K) {
      const bool deep = FMT == FMT_Q6_K || (S >= 2 * NW && rounds(2) >= 2);
      if (deep && t22 < t1) {
        go(kquant_gemv_mt<FMT, NW, 2, 2>, 2, 2);
        SV_CHECK_LAUNCH();
        return SV_OK;
      }
    }
  }
  if (two) go(kquant_gemv_mt<FMT, NW, 1, 2>, 1, 2);
  else go(kquant_gemv_mt<FMT, NW, 1, 1>, 1, 1);
  SV_CHECK_LAUNCH();
  return SV_OK;
}

// ---------------------------------------------------------------------------------------
// Repack GGUF blocks into (quant, meta).
// ---------------------------------------------------------------------------------------
// Rows n >= n_split come from `bottom` (row n - n_split), so that two GGUF tensors of one
// format repack as one matrix ([gate; up] of an expert); single matrices pass n_split = N.
__device__ __forceinline__ const uint8_t* src_block(const uint8_t* top, const uint8_t* bottom,
                                                    int64_t n_split, int64_t n, int64_t s,
                                                    int64_t S, int64_t bytes) {
  return n < n_split ? top + (n * S + s) * bytes : bottom + ((n - n_split) * S + s) * bytes;
}

__global__ void shuffle_q4k(const uint8_t* __restrict__ gguf, const uint8_t* __restrict__ gguf2,
                            int64_t n_split, uint8_t* __restrict__ quant,
                            uint8_t* __restrict__ meta, int64_t N, int64_t S) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= N * S) return;
  const int64_t n = id / S, s = id % S;
  const uint8_t* blk = src_block(gguf, gguf2, n_split, n, s, S, 144);
  const int64_t tile = n / TILE_N;
  const int col = (int)(n % TILE_N);
  const int64_t ts = tile * S + s;
  uint8_t* mo = meta + (ts * 16 + col) * 16;
  for (int i = 0; i < 16; ++i) mo[i] = blk[i];
  const uint8_t* qs = blk + 16;
  for (int h = 0; h < 2; ++h)
    for (int kq = 0; kq < 4; ++kq) {
      const int lane = col + 16 * kq;
      uint8_t* qo = quant + ((ts * 2 + h) * 64 + lane) * 16;
      for (int i = 0; i < 8; ++i) {
        qo[i] = qs[64 * h + 8 * kq + i];
        qo[8 + i] = qs[64 * h + 32 + 8 * kq + i];
      }
    }
}

__global__ void shuffle_q80(const uint8_t* __restrict__ gguf, const uint8_t* __restrict__ gguf2,
                            int64_t n_split, uint8_t* __restrict__ quant,
                            uint8_t* __restrict__ meta, int64_t N, int64_t S) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= N * S) return;
  const int64_t n = id / S, s = id % S;
  const int64_t tile = n / TILE_N;
  const int col = (int)(n % TILE_N);
  const int64_t ts = tile * S + s;
  for (int j = 0; j < 8; ++j) {
    const uint8_t* blk = src_block(gguf, gguf2, n_split, n, s, S, 8 * 34) + j * 34;
    uint8_t* mo = meta + (ts * 16 + col) * 16 + 2 * j;
    mo[0] = blk[0];
    mo[1] = blk[1];
    const int jp = j >> 1, half = j & 1;
    for (int kq = 0; kq < 4; ++kq) {
      const int lane = col + 16 * kq;
      uint8_t* qo = quant + ((ts * 4 + jp) * 64 + lane) * 16 + 8 * half;
      for (int i = 0; i < 8; ++i) qo[i] = blk[2 + 8 * kq + i];
    }
  }
}

// Q5_K: the Q4_K nibble layout of qs (@48), then each lane's 8 qh bytes (@16) after the tile-
// superblock's nibbles; meta as Q4_K (d, dmin, scales: the block's first 16 bytes).
__global__ void shuffle_q5k(const uint8_t* __restrict__ gguf, const uint8_t* __restrict__ gguf2,
                            int64_t n_split, uint8_t* __restrict__ quant,
                            uint8_t* __restrict__ meta, int64_t N, int64_t S) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= N * S) return;
  const int64_t n = id / S, s = id % S;
  const uint8_t* blk = src_block(gguf, gguf2, n_split, n, s, S, 176);
  const int64_t tile = n / TILE_N;
  const int col = (int)(n % TILE_N);
  const int64_t ts = tile * S + s;
  uint8_t* mo = meta + (ts * 16 + col) * 16;
  for (int i = 0; i < 16; ++i) mo[i] = blk[i];
  const uint8_t* qh = blk + 16;
  const uint8_t* qs = blk + 48;
  uint8_t* base = quant + ts * 2560;
  for (int kq = 0; kq < 4; ++kq) {
    const int lane = col + 16 * kq;
    for (int h = 0; h < 2; ++h) {
      uint8_t* qo = base + (h * 64 + lane) * 16;
      for (int i = 0; i < 8; ++i) {
        qo[i] = qs[64 * h + 8 * kq + i];
        qo[8 + i] = qs[64 * h + 32 + 8 * kq + i];
      }
    }
    uint8_t* ho = base + 2048 + lane * 8;
    for (int i = 0; i < 8; ++i) ho[i] = qh[8 * kq + i];
  }
}

// Q6_K: per lane three 16-byte vectors (ql of half 0, ql of half 1, qh of both halves, each
// the bytes l = 8 kq .. 8 kq + 7 of its two 32-byte runs); meta: the 16 int8 scales per
// column, and after every tile-superblock's scales the fp16 d per (tile-superblock, column).
__global__ void shuffle_q6k(const uint8_t* __restrict__ gguf, const uint8_t* __restrict__ gguf2,
                            int64_t n_split, uint8_t* __restrict__ quant,
                            uint8_t* __restrict__ meta, int64_t N, int64_t S) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= N * S) return;
  const int64_t n = id / S, s = id % S;
  const uint8_t* blk = src_block(gguf, gguf2, n_split, n, s, S, 210);
  const int64_t tile = n / TILE_N;
  const int col = (int)(n % TILE_N);
  const int64_t ts = tile * S + s;
  uint8_t* mo = meta + (ts * 16 + col) * 16;
  for (int i = 0; i < 16; ++i) mo[i] = blk[192 + i];
  uint8_t* dd = meta + N * S * 16 + (ts * 16 + col) * 2;
  dd[0] = blk[208];
  dd[1] = blk[209];
  const uint8_t* ql = blk;
  const uint8_t* qh = blk + 128;
  uint8_t* base = quant + ts * 3072;
  for (int kq = 0; kq < 4; ++kq) {
    const int lane = col + 16 * kq;
    for (int half = 0; half < 2; ++half) {
      uint8_t* qo = base + (half * 64 + lane) * 16;
      for (int i = 0; i < 8; ++i) {
        qo[i] = ql[64 * half + 8 * kq + i];
        qo[8 + i] = ql[64 * half + 32 + 8 * kq + i];
      }
    }
    uint8_t* ho = base + (2 * 64 + lane) * 16;
    for (int i = 0; i < 8; ++i) {
      ho[i] = qh[8 * kq + i];
      ho[8 + i] = qh[32 + 8 * kq + i];
    }
  }
}

bool fmt_ok(int fmt) {
  return fmt == FMT_Q4_K || fmt == FMT_Q5_K || fmt == FMT_Q6_K || fmt == FMT_Q8_0;
}

// The GEMV kernels address a weight through one buffer resource with 32-bit offsets: its
// packed quants (N * K / 2 bytes for Q4_K, N * K for Q8_0) must stay below 4 GiB.
bool weight_fits(int fmt, int64_t N, int64_t K) {
  const int64_t qbytes = fmt == FMT_Q4_K ? N * (K / 2) : fmt == FMT_Q5_K ? N * (K / 256) * 160
                         : fmt == FMT_Q6_K ? N * (K / 256) * 192 : N * K;
  return qbytes <= (int64_t)0xFFFFFC00 && N * (K / 256) * 256 <= (int64_t)0xFFFFFFFF;
}

template <int FMT, int NTILE, int NW, bool RAW = false>
int launch_gemv(const void* quant, const void* meta, const void* ws, void* c, int M, int N, int S,
                int c_bf16, int ldc, hipStream_t s) {
  const int tiles = N / TILE_N;
  const int grid = (tiles + NTILE - 1) / NTILE;
  hipLaunchKernelGGL((kquant_gemv<FMT, NTILE, NW, RAW>), dim3(grid), dim3(NW * 64), 0, s,
                     (const u32x4*)quant, (const u32x4*)meta, ws, c, M, N, S, c_bf16, ldc);
  SV_CHECK_LAUNCH();
  return SV_OK;
}

int g_gemv_variant = 0;  // 0 = automatic; see snowverify_gemv_variant

// Calls f with std::integral_constant<int, FMT> for a supported format id.
template <class F>
int by_format(int fmt, F&& f) {
  switch (fmt) {
    case FMT_Q4_K: return f(std::integral_constant<int, FMT_Q4_K>{});
    case FMT_Q5_K: return f(std::integral_constant<int, FMT_Q5_K>{});
    case FMT_Q6_K: return f(std::integral_constant<int, FMT_Q6_K>{});
    case FMT_Q8_0: return f(std::integral_constant<int, FMT_Q8_0>{});
    default: return SV_EINVAL;
  }
}

template <int FMT, bool RAW = false>
int dispatch_gemv(const void* quant, const void* meta, const void* ws, void* c, int M, int N,
                  int S, int c_bf16, int ldc, hipStream_t s) {
  switch (g_gemv_variant) {
    case 1: return launch_gemv<FMT, 1, 4, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    case 2: return launch_gemv<FMT, 2, 4, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    case 3: return launch_gemv<FMT, 4, 4, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    case 4: return launch_gemv<FMT, 1, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    case 5: return launch_gemv<FMT, 2, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    case 6: return launch_gemv<FMT, 4, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    default: break;
  }
  const int tiles = N / TILE_N;
  // measured on MI355X (M = 9): wide outputs want 4 tiles x 8 waves, K >= 4096 narrow outputs
  // 1 x 8, K = 2048 2 x 8 when there are >= 2 tiles per CU, K = 4096 (prepared operands)
  // 2 x 8 from 3 tiles per CU (6144 x 4096: 9.7 -> 7.6 us)
  if (S >= 8) {
    // (Q8_0 keeps two tiles: four tiles of int8 quants exceed the register file)
    if (tiles >= 4 * 192 && FMT == FMT_Q4_K)
      return launch_gemv<FMT, 4, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    if (tiles >= 2 * 128 && S <= 8) return launch_gemv<FMT, 2, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    if (!RAW && FMT == FMT_Q4_K && tiles >= 3 * 128 && S <= 16)
      return launch_gemv<FMT, 2, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
    return launch_gemv<FMT, 1, 8, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
  }
  if (tiles >= 2 * 256) return launch_gemv<FMT, 2, 4, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
  return launch_gemv<FMT, 1, 4, RAW>(quant, meta, ws, c, M, N, S, c_bf16, ldc, s);
}

}  // namespace

// =======================================================================================
// C ABI
// =======================================================================================

SV_API int64_t snowllm_kquant_gguf_bytes(int fmt, int64_t N, int64_t K) {
  if (N < 0 || K < 0) return -1;
  if (fmt == FMT_Q4_K) return K % 256 ? -1 : N * (K / 256) * 144;
  if (fmt == FMT_Q5_K) return K % 256 ? -1 : N * (K / 256) * 176;
  if (fmt == FMT_Q6_K) return K % 256 ? -1 : N * (K / 256) * 210;
  if (fmt == FMT_Q8_0) return K % 32 ? -1 : N * (K / 32) * 34;
  return -1;
}

// Repacked sizes: quant + meta - 4 = the GGUF bytes (the quant buffer keeps 4 bytes of slack).
SV_API int64_t snowllm_kquant_quant_bytes(int fmt, int64_t N, int64_t K) {
  if (!fmt_ok(fmt) || N < 0 || K % 256 || N % TILE_N) return -1;
  const int64_t blocks = N * (K / 256);
  switch (fmt) {
    case FMT_Q4_K: return blocks * 128 + 4;
    case FMT_Q5_K: return blocks * 160 + 4;
    case FMT_Q6_K: return blocks * 192 + 4;
    default: return N * K + 4;
  }
}

SV_API int64_t snowllm_kquant_meta_bytes(int fmt, int64_t N, int64_t K) {
  if (!fmt_ok(fmt) || N < 0 || K % 256 || N % TILE_N) return -1;
  return N * (K / 256) * (fmt == FMT_Q6_K ? 18 : 16);
}

SV_API int snowllm_kquant_supported(int fmt) { return fmt_ok(fmt) ? 1 : 0; }

// Extension (tuning knob, no counterpart in the reference): force a GEMV tile shape
// (0 = automatic, 1..6 = fixed (tiles per workgroup, waves) pairs). Process-global.
SV_API void snowverify_gemv_variant(int v) { g_gemv_variant = v; }

// Extension (no counterpart in the reference): repack two GGUF tensors of one format, `top`
// (rows 0 .. n_top - 1) and `bottom` (rows n_top .. N - 1), as one [N, K] matrix -- an
// expert's [gate; up] from its two stacks.
SV_API int snowverify_kquant_shuffle_split(int fmt, const uint8_t* top, const uint8_t* bottom,
                                           int64_t n_top, uint8_t* quant, uint8_t* meta,
                                           int64_t N, int64_t K, void* stream) {
  if (!fmt_ok(fmt) || N <= 0 || K <= 0 || K % 256 || N % TILE_N || n_top < 0 || n_top > N ||
      !top || (n_top < N && !bottom))
    return SV_EINVAL;
  const int64_t S = K / 256;
  const int64_t total = N * S;
  const int nt = 256;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)((total + nt - 1) / nt));
  if (fmt == FMT_Q4_K)
    hipLaunchKernelGGL(shuffle_q4k, grid, dim3(nt), 0, s, top, bottom, n_top, quant, meta, N, S);
  else if (fmt == FMT_Q5_K)
    hipLaunchKernelGGL(shuffle_q5k, grid, dim3(nt), 0, s, top, bottom, n_top, quant, meta, N, S);
  else if (fmt == FMT_Q6_K)
    hipLaunchKernelGGL(shuffle_q6k, grid, dim3(nt), 0, s, top, bottom, n_top, quant, meta, N, S);
  else
    hipLaunchKernelGGL(shuffle_q80, grid, dim3(nt), 0, s, top, bottom, n_top, quant, meta, N, S);
  SV_CHECK_LAUNCH();
  return SV_OK;
}

SV_API int snowllm_gemm_kquant_shuffle_b(int fmt, const uint8_t* gguf, uint8_t* quant,
                                         uint8_t* meta, int64_t N, int64_t K, void* stream) {
  return snowverify_kquant_shuffle_split(fmt, gguf, nullptr, N, quant, meta, N, K, stream);
}

SV_API int64_t snowllm_gemm_kquant_a_ws_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % 256) return 0;
  const int64_t tiles = (M + TILE_M - 1) / TILE_M;
  return (int64_t)(tiles * xprep_tile_bytes(K / 256));
}

// Extension (no counterpart in the reference): convert activations once into the operand
// workspace so several weights that share an input (gate/up, Q/K/V) reuse it.
SV_API int snowverify_gemm_kquant_prepare_a(const void* a, int64_t M, int64_t K, void* ws,
                                         void* stream) {
  if (M < 0 || K <= 0 || K % 256) return SV_EINVAL;
  if (M == 0) return SV_OK;
  const int64_t S = K / 256;
  const int64_t mt = (M + TILE_M - 1) / TILE_M;
  hipLaunchKernelGGL(xprep_kernel, dim3((unsigned)S, (unsigned)mt), dim3(64), 0,
                     (hipStream_t)stream, (const uint16_t*)a, M, K, ws, xprep_tile_bytes(S));
  SV_CHECK_LAUNCH();
  return SV_OK;
}

// Extension (no counterpart in the reference): the GEMV on a prepared operand workspace,
// writing row m of the result at c + m * ldc (ldc >= N elements), so that two weights of
// different formats fill the column ranges of one output (Q|K and V of a fused projection).
SV_API int snowverify_gemm_kquant_a_prepared_ld(int fmt, const uint8_t* quant,
                                                const uint8_t* meta, void* c, int64_t ldc,
                                                int64_t M, int64_t N, int64_t K, int c_is_bf16,
                                                const void* ws, void* stream) {
  if (!fmt_ok(fmt) || M < 0 || N <= 0 || K <= 0 || K % 256 || N % TILE_N || ldc < N ||
      ldc > INT32_MAX)
    return SV_EINVAL;
  if (!weight_fits(fmt, N, K)) return SV_ENOTSUP;
  if (M == 0) return SV_OK;
  hipStream_t s = (hipStream_t)stream;
  const int64_t S = K / 256;
  const size_t tb = xprep_tile_bytes(S);
  const int64_t mt = (M + TILE_M - 1) / TILE_M;
  const size_t esz = c_is_bf16 ? 2 : 4;
  const int ld = (int)ldc;
  if (mt > 1 && g_gemv_variant == 0) {
    // wider than one row tile: one launch over every row tile (the waves split the
    // superblocks as the automatic 16-row launch does: the same bits)
    return by_format(fmt, [&](auto F) {
      constexpr int FM = decltype(F)::value;
      return S >= 8 ? launch_gemv_mt<FM, 8>(quant, meta, ws, c, (int)M, (int)N, (int)S, c_is_bf16, ld, s)
                    : launch_gemv_mt<FM, 4>(quant, meta, ws, c, (int)M, (int)N, (int)S, c_is_bf16, ld, s);
    });
  }
  for (int64_t t = 0; t < mt; ++t) {
    const int rows = (int)((M - t * TILE_M) < TILE_M ? (M - t * TILE_M) : TILE_M);
    void* ct = (char*)c + (size_t)t * TILE_M * ldc * esz;
    const void* wst = (const char*)ws + t * tb;
    int rc = by_format(fmt, [&](auto F) {
      return dispatch_gemv<decltype(F)::value>(quant, meta, wst, ct, rows, (int)N, (int)S,
                                               c_is_bf16, ld, s);
    });
    if (rc) return rc;
  }
  return SV_OK;
}

// Extension (no counterpart in the reference): the GEMV on a prepared operand workspace.
SV_API int snowverify_gemm_kquant_a_prepared(int fmt, const uint8_t* quant, const uint8_t* meta,
                                          void* c, int64_t M, int64_t N, int64_t K,
                                          int c_is_bf16, const void* ws, void* stream) {
  return snowverify_gemm_kquant_a_prepared_ld(fmt, quant, meta, c, N, M, N, K, c_is_bf16, ws,
                                              stream);
}

SV_API int snowllm_gemm_kquant_a(int fmt, const void* a, const uint8_t* quant, const uint8_t* meta,
                                 void* c, int64_t M, int64_t N, int64_t K, int c_is_bf16, void* ws,
                                 void* stream) {
  if (!fmt_ok(fmt) || M < 0 || N <= 0 || K <= 0 || K % 256 || N % TILE_N) return SV_EINVAL;
  if (!weight_fits(fmt, N, K)) return SV_ENOTSUP;
  if (M == 0) return SV_OK;
  if (M <= TILE_M && M * K * 2 <= INT32_MAX) {
    // one launch: the GEMV converts the bf16 activations itself (same operands as the
    // prepared path, so the same results); ws is not touched
    hipStream_t s = (hipStream_t)stream;
    return by_format(fmt, [&](auto F) {
      return dispatch_gemv<decltype(F)::value, true>(quant, meta, a, c, (int)M, (int)N,
                                                     (int)(K / 256), c_is_bf16, (int)N, s);
    });
  }
  int rc = snowverify_gemm_kquant_prepare_a(a, M, K, ws, stream);
  if (rc) return rc;
  return snowverify_gemm_kquant_a_prepared(fmt, quant, meta, c, M, N, K, c_is_bf16, ws, stream);
}

// ---------------------------------------------------------------------------------------
// The no-allocation form of snowllm_gemm_kquant_a, for callers that cannot allocate (code
// under HIP-graph capture, tight serving loops, harnesses that forbid hipMalloc). Up to 16
// rows the GEMV converts the activations itself and needs no workspace; above that the
// operand workspace lives in `scratch`, a file-scope device array of a fixed size -- each GPU
// the library runs on holds its own copy until the process ends. Host code never passes the
// array's name to a kernel: its device address is read once per device with
// hipGetSymbolAddress, with that device current, and kept.
// ---------------------------------------------------------------------------------------
namespace {
constexpr int64_t NOALLOC_MAX_M = 64, NOALLOC_MAX_K = 16384;
constexpr size_t NOALLOC_WS_BYTES = 2244608;  // snowllm_gemm_kquant_a_ws_bytes(64, 16384)
static __device__ __align__(256) uint8_t scratch[NOALLOC_WS_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[MAX_DEVICES];

// The current device's address of `scratch`.
int scratch_address(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= MAX_DEVICES) return SV_ENOTSUP;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return SV_EINVAL;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return SV_OK;
}
}  // namespace

SV_API int snowverify_gemm_kquant_a_noalloc(int fmt, const void* a, const uint8_t* quant,
                                            const uint8_t* meta, void* c, int64_t M, int64_t N,
                                            int64_t K, int c_is_bf16, void* stream) {
  if (!fmt_ok(fmt) || M < 0 || N <= 0 || K <= 0 || K % 256 || N % TILE_N) return SV_EINVAL;
  if (M > NOALLOC_MAX_M || K > NOALLOC_MAX_K) return SV_EINVAL;  // beyond the array
  if (M == 0) return SV_OK;
  if (M <= TILE_M)  // the one-launch form: no workspace
    return snowllm_gemm_kquant_a(fmt, a, quant, meta, c, M, N, K, c_is_bf16, nullptr, stream);
  if ((size_t)snowllm_gemm_kquant_a_ws_bytes(M, K) > NOALLOC_WS_BYTES) return SV_EINVAL;
  void* ws = nullptr;
  int rc = scratch_address(&ws);
  if (rc) return rc;
  // the prep pass writes every byte of the workspace the GEMV reads (padding rows included),
  // so nothing needs clearing between calls
  rc = snowverify_gemm_kquant_prepare_a(a, M, K, ws, stream);
  if (rc) return rc;
  return snowverify_gemm_kquant_a_prepared(fmt, quant, meta, c, M, N, K, c_is_bf16, ws, stream);
}
