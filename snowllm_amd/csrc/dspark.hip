// The DSpark Markov head (snowllm/ops/dspark.py:10-16, 53-77; snowllm/_capi.py:567-573): a
// greedy walk over a draft block in which every row's logits get a low-rank bias from the
// previous token,
//
//   latent = W1[prev]                       (prev = the anchor, then the previous row's pick)
//   bias   = W2 latent                      (one value per vocabulary row)
//   pick   = argmax fp32(base + bias)        confidence = sigmoid([hidden, latent] . w + b)
//
// (the reference's PyTorch restatement: tests/test_lfm2_dspark_reference.py:143-152).
//
// Each row streams all of W2 ([V, rank] bf16, 78 MB at V = 151936, rank 256) once for every
// request of the batch together, one launch per block row. The bias that counts is the sum of
// the bf16 products taken in fp64 -- exact -- and rounded once, but only the largest score is
// wanted: 16 rows x 16 requests at a time the matrix cores give every bias in fp32 with a bound
// on its error (from the sum of the products' magnitudes, a second product), hence bounds on
// every score, and only rows whose upper bound reaches the largest lower bound seen (a few per
// workgroup, usually one per request in all) are summed in fp64. W2 is packed in tiles of 64
// rows, 8 values of a row per 16 bytes, so that a 16-row operand of 32 values is four runs of
// 256 bytes. Every workgroup reduces its rows to one (value, index) key per request; the last
// workgroup of a two-level arrival reduces the keys and writes the pick, which the next row's
// launch reads as its latent index; one more workgroup computes the confidences.
// Bound: the read of W2, from the 256 MB cache after the first row, and below about 50 MB the
// chain of the row (the latent's read, the bounds, the exact sum of the workgroup's best row, the
// two arrivals). Sharing the lower bound between workgroups was slower for up to eight requests
// (its round trip costs what it saves). MI355X, us per block row with confidences, every sum in
// fp64 before -> now: V = 151,936, rank 256: 29 -> 21 for one request, 45 -> 25 for four, 108 ->
// 31 for eight, 187 -> 46 for sixteen; rank 64: 14.8 -> 14.5, 26 -> 17.5, 57 -> 21 for one, four,
// eight; V = 32,000, rank 256: 19 -> 15, 33 -> 17, 61 -> 23. Masked logits (-inf, or the type's
// lowest value) 45 -> 24 at four requests. Equal scores everywhere (a W2 of zeros under constant
// logits) need every row's exact sum behind the bounds: 29 -> 33, 45 -> 58 and 184 -> 116 for one,
// four and sixteen requests, where a wave per row took 95, 290 and 1090.
#include "common.h"

namespace {

constexpr int DSP_WAVES = 4;               // waves per workgroup, 16 rows each at a time
constexpr int DSP_NT = DSP_WAVES * WAVE;
constexpr int DSP_MAX_B = 16;              // requests per call
constexpr int DSP_MAX_RANK = 512;
constexpr uint64_t DSP_QUANTUM = 1ull << 20;  // > workgroups of a launch
constexpr int64_t DSP_MAX_V = (int64_t)1 << 31;

// Arrivals of the last launch (library-owned; calls on one device are stream-ordered). Each
// launch adds exactly one quantum, so the count stays a multiple of it between launches and
// captured replays need no reset.
__device__ uint64_t g_dsp_cnt;

// Packed W2: tile t holds rows [64 t, 64 t + rows_t), rows_t = min(64, n - 64 t), and stores
// chunk c (elements 8c .. 8c + 7) of its rows at elements 64 t k + (c rows_t + lane) 8. The
// packed matrix has exactly the n k elements of the source.
__global__ void dsp_pack_kernel(const uint16_t* __restrict__ raw, uint16_t* __restrict__ packed,
                                int64_t n, int64_t k) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;   // 16-byte chunk of the source
  const int64_t chunks = k / 8;
  if (i >= n * chunks) return;
  const int64_t row = i / chunks, c = i % chunks;
  const int64_t t = row / 64, lane = row % 64;
  const int64_t rows_t = n - 64 * t < 64 ? n - 64 * t : 64;
  const uint4 v = *(const uint4*)(raw + row * k + c * 8);
  *(uint4*)(packed + 64 * t * k + (c * rows_t + lane) * 8) = v;
}

// fp64 -> the nearest bf16 value, rounded once: round to odd at fp32 (16 spare bits), then to
// nearest-even at bf16.
__device__ __forceinline__ float bf16_from_f64(double d) {
  const float t = (float)d;
  uint32_t u = __float_as_uint(t);
  if ((double)t != d && d == d) {
    if (fabs((double)t) > fabs(d)) u -= 1;  // the fp32 rounding went away from zero: step back
    u |= 1;
  }
  return bf16_to_f32(f32_to_bf16(__uint_as_float(u)));
}

struct DspArgs {
  const float* base;        // [b * block, base_stride] f32
  const uint16_t* w1;       // [v, rank] bf16
  const uint16_t* w2;       // packed [v, rank] bf16
  const int64_t* anchor;    // [b]
  const uint16_t* pre_head; // [b * block, ps] bf16 or null
  const float* conf_w;      // [h + rank]
  const float* conf_b;      // scalar or null
  int64_t* out;             // [b, block]
  float* confidence;        // [b, block] or null
  uint64_t* partial;        // [b, nwg]
  int64_t v, base_stride, ps;
  int b, rank, block, h, nwg, fp32_bias, j;
};

// Grid: G <= 1024 workgroups of 4 waves; wave k of workgroup g takes the 16-row units 4 g + k,
// 4 g + k + 4 G, ... with the next unit's operands in flight.
// Arrival is two-level so that no counter sees more than 32 arrivals: the workgroups of a
// group of 32 count on the group's counter; the group's last arrival reduces the group's keys
// and counts on the top counter, whose last arrival reduces the groups' keys and writes the
// pick.
constexpr int DSP_GRID = 1024, DSP_GROUP = 32, DSP_GROUPS = DSP_GRID / DSP_GROUP;
__device__ uint64_t g_dsp_group[DSP_GROUPS];

__device__ __forceinline__ bool dsp_arrive(uint64_t* cnt, int n, bool lead, uint32_t* s_flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's stores have completed
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint64_t inc = lead ? DSP_QUANTUM - (uint64_t)n + 1 : 1;
    const uint64_t old = __hip_atomic_fetch_add(cnt, inc, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    *s_flag = ((old + inc) & (DSP_QUANTUM - 1)) == 0;
  }
  __syncthreads();
  return *s_flag != 0;
}

__device__ __forceinline__ uint64_t dsp_load(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The exact score of one vocabulary row for one request (L: its latent in fp32), by one wave: a
// chunk of eight products per lane in fp64, the lanes' sums added (exact in any order), the
// sum rounded once. The key in every lane.
__device__ __forceinline__ uint64_t dsp_exact_key(const DspArgs& a, const float* L, int r,
                                                  int64_t row) {
  const int chunks = a.rank / 8, lane = threadIdx.x & (WAVE - 1);   // chunks <= 64
  const int64_t tile = row / WAVE;
  const int64_t rows_t = a.v - tile * WAVE < WAVE ? a.v - tile * WAVE : WAVE;
  const uint4* src = (const uint4*)(a.w2 + tile * WAVE * (int64_t)a.rank) + row % WAVE;
  const int c = lane < chunks ? lane : 0;
  const uint4 q = src[c * rows_t];
  const float x = a.base[((int64_t)r * a.block + a.j) * a.base_stride + row];
  const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
  double acc = 0.0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float* l = L + c * 8 + 2 * e;
    acc += (double)(__uint_as_float(qw[e] << 16) * l[0]);        // exact bf16 x bf16
    acc += (double)(__uint_as_float(qw[e] & 0xffff0000u) * l[1]);
  }
  if (lane >= chunks) acc = 0.0;
#pragma unroll
  for (int d = WAVE / 2; d > 0; d >>= 1)
    acc += __builtin_bit_cast(double, shfl_xor_u64(__builtin_bit_cast(uint64_t, acc), d));
  const float bias = a.fp32_bias ? (float)acc : bf16_from_f64(acc);
  return argmax_key(x + bias, (uint32_t)row);
}

// The same scores by one lane, of one row for NR requests r0, r0 + 1, ... (those from B on come out
// as r0's), for many candidates: rows may differ from lane to lane, and neighbouring rows are
// neighbouring words of the packed tile. The next chunks load behind the sums.
template <int NR>
__device__ __forceinline__ void dsp_lane_keys(const DspArgs& a, const float* s_lat, int r0,
                                              int64_t row, uint64_t (&key)[NR]) {
  const int chunks = a.rank / 8;
  const int64_t tile = row / WAVE;
  const int64_t rows_t = a.v - tile * WAVE < WAVE ? a.v - tile * WAVE : WAVE;
  const uint4* src = (const uint4*)(a.w2 + tile * WAVE * (int64_t)a.rank) + row % WAVE;
  const float* L[NR];
  float x[NR];
  double acc[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = r0 + i < a.b ? r0 + i : r0;
    L[i] = s_lat + r * a.rank;
    x[i] = a.base[((int64_t)r * a.block + a.j) * a.base_stride + row];
    acc[i] = 0.0;
  }
  constexpr int UN = 4;  // chunks of a load
  uint4 q[2][UN];
  auto load = [&](int b, int cb) {
#pragma unroll
    for (int u = 0; u < UN; ++u) q[b][u] = src[(cb + u < chunks ? cb + u : chunks - 1) * rows_t];
  };
  auto sum = [&](int b, int cb) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (cb + u >= chunks) break;  // uniform
      const uint32_t qw[4] = {q[b][u].x, q[b][u].y, q[b][u].z, q[b][u].w};
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        double s0 = 0.0, s1 = 0.0;  // two chains; the sum stays exact
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float* l = L[i] + (cb + u) * 8 + 2 * e;
          s0 += (double)(__uint_as_float(qw[e] << 16) * l[0]);
          s1 += (double)(__uint_as_float(qw[e] & 0xffff0000u) * l[1]);
        }
        acc[i] += s0 + s1;
      }
    }
  };
  load(0, 0);
  for (int cb = 0; cb < chunks; cb += 2 * UN) {
    load(1, cb + UN);
    sum(0, cb);
    load(0, cb + 2 * UN);
    sum(1, cb + UN);
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const float bias = a.fp32_bias ? (float)acc[i] : bf16_from_f64(acc[i]);
    key[i] = argmax_key(x[i] + bias, (uint32_t)row);
  }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int DSP_UNIT = 16;              // vocabulary rows of a matrix product
constexpr int DSP_CAND = 512;             // candidates a workgroup keeps
constexpr int DSP_FEW = 32;               // candidates up to here are looked at in turn
constexpr uint32_t DSP_BOTTOM = 0x007fffffu;  // ord_key(-inf)

// KS: 32-value steps of the rank (values past the rank are zero operands).
template <int KS>
__global__ void __launch_bounds__(DSP_NT) dsp_markov_kernel(DspArgs a) {
  __shared__ float s_lat[4096];                  // latents f32 [b][rank], b rank <= 4096
  __shared__ uint64_t s_best[DSP_MAX_B];
  __shared__ uint32_t s_low[DSP_MAX_B];          // this workgroup's largest lower bound
  __shared__ uint32_t s_up[DSP_CAND];            // candidates: upper bound (key), row, request
  __shared__ uint32_t s_row[DSP_CAND];
  __shared__ uint8_t s_req[DSP_CAND];
  __shared__ uint16_t s_left[DSP_CAND];          // candidates that every wave's bounds leave
  __shared__ uint32_t s_n, s_m, s_flag;
  const int t = threadIdx.x, lane = t & (WAVE - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / WAVE);
  const int B = a.b, R = a.rank, j = a.j, G = a.nwg;
  const int col = lane & 15, kq = lane >> 4, chunks = R / 8;
  const int64_t units = (a.v + DSP_UNIT - 1) / DSP_UNIT;
  // operand chunks 4 s + kq of the unit's rows (the tile as the buffer: chunks past the rank, rows
  // past the vocabulary and units past the last are out of its range and read zeros without
  // touching memory; the whole offset is the vector one, which the bounds check covers) and the
  // unit's base logits
  auto load_unit = [&](int64_t u, uint4 (&q)[KS], float (&x)[4]) {
    const int64_t tile = u * DSP_UNIT / WAVE;
    const int64_t left = a.v - tile * WAVE;
    const int rows_t = left >= WAVE ? WAVE : left > 0 ? (int)left : 0;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.w2 + (rows_t ? tile * WAVE * (int64_t)R : 0)), 0, u < units ? rows_t * R * 2 : 0,
        0x00020000);
    const uint32_t at = (uint32_t)((kq * rows_t + (int)(u * DSP_UNIT % WAVE) + col) * 16);
#pragma unroll
    for (int s = 0; s < KS; ++s)
      q[s] = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(wr, at + (uint32_t)(4 * s * rows_t * 16), 0, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t n = u * DSP_UNIT + 4 * kq + i;
      x[i] = a.base[((int64_t)(col < B ? col : 0) * a.block + j) * a.base_stride +
                    (n < a.v ? n : a.v - 1)];
    }
  };
  if ((int)blockIdx.x == G) {
    // one workgroup more when confidences are wanted: they need the row's latent, not its pick
    for (int r = w; r < B; r += DSP_WAVES) {
      const int64_t at = (int64_t)r * a.block + j;
      const int64_t prev = j == 0 ? a.anchor[r] : a.out[at - 1];
      const uint16_t* lt = prev >= 0 && prev < a.v ? a.w1 + prev * R : nullptr;
      const uint16_t* hid = a.pre_head + at * a.ps;
      float z = 0.f;
#pragma unroll 16
      for (int i = lane; i < a.h; i += WAVE) z += bf16_to_f32(hid[i]) * a.conf_w[i];
      for (int i = lane; i < R; i += WAVE) z += (lt ? bf16_to_f32(lt[i]) : 0.f) * a.conf_w[a.h + i];
      z = wave_sum(z);
      if (lane == 0) {
        if (a.conf_b) z += *a.conf_b;
        a.confidence[at] = 1.f / (1.f + expf(-z));
      }
    }
    return;
  }
  int64_t u = (int64_t)blockIdx.x * DSP_WAVES + w;
  uint4 q0[KS], q1[KS];
  float x0[4], x1[4];
  load_unit(u, q0, x0);
  // (a workgroup's first row scores -inf at least: the result where every score is -inf)
  if (t < DSP_MAX_B) {
    s_low[t] = 0u;
    s_best[t] = argmax_key(-__builtin_huge_valf(), (uint32_t)(blockIdx.x * DSP_WAVES * DSP_UNIT));
  }
  if (t == 0) s_n = s_m = 0u;
  for (int i = t; i < B * R; i += DSP_NT) {
    const int r = i / R, e = i % R;
    const int64_t prev = j == 0 ? a.anchor[r] : a.out[(int64_t)r * a.block + j - 1];
    s_lat[i] = (prev >= 0 && prev < a.v) ? bf16_to_f32(a.w1[prev * R + e]) : 0.f;
  }
  __syncthreads();
  // the requests' latents as the other operand (column col: request col)
  bf16x8 lat[KS];
  float top = 0.f;
  bool subnormal = false;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    uint32_t l[4] = {0u, 0u, 0u, 0u};
    if (col < B && 4 * s + kq < chunks)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float* f = s_lat + col * R + (4 * s + kq) * 8 + 2 * e;
        l[e] = (__float_as_uint(f[0]) >> 16) | (__float_as_uint(f[1]) & 0xffff0000u);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float m = __builtin_fabsf(f[k]);
          top = m > top ? m : top;
          subnormal |= m > 0.f && m < 1.17549435e-38f;
        }
      }
    lat[s] = __builtin_bit_cast(bf16x8, uint4{l[0], l[1], l[2], l[3]});
  }

  // |fp32 sum - exact sum| <= err Sabs: every addition of the matrix cores' chain rounds by at
  // most 2^-22 of the running magnitude (twice a binary32 ulp, whatever the order and the
  // rounding), products are exact; tiny covers products and sums below the normal range, and
  // weights there, should the cores take them as zero (latents there: every row is a candidate)
  const float err = (float)(R + 8) * 2.384185791015625e-07f;
  top = fmaxf(top, __shfl_xor(top, 16, WAVE));
  top = fmaxf(top, __shfl_xor(top, 32, WAVE));
  const uint64_t sub = __ballot(subnormal);
  const float tiny = (sub >> col & 0x0001000100010001ull)
                         ? __builtin_huge_valf() : 1e-30f + (float)R * 1.17549435e-38f * top;
  // rounding of the bias (bf16: 2^-9 to nearest, stated as 2^-8) and of the score in fp32
  const float rnd = a.fp32_bias ? 2.384185791015625e-07f : 3.90625e-03f, ulp = 2.384185791015625e-07f;
  uint32_t low = 0u;  // this lane's request: the largest lower bound of the wave's rows
  uint64_t known = 0ull;  // and its best row whose score is known
  for (; u < units; u += (int64_t)G * DSP_WAVES) {
    load_unit(u + (int64_t)G * DSP_WAVES, q1, x1);
    floatx4 c = {0.f, 0.f, 0.f, 0.f}, ca = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4 qa = {q0[s].x & 0x7fff7fffu, q0[s].y & 0x7fff7fffu, q0[s].z & 0x7fff7fffu,
                        q0[s].w & 0x7fff7fffu};
      const uint4 lw = __builtin_bit_cast(uint4, lat[s]);
      const uint4 la = {lw.x & 0x7fff7fffu, lw.y & 0x7fff7fffu, lw.z & 0x7fff7fffu, lw.w & 0x7fff7fffu};
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, q0[s]), lat[s], c, 0, 0, 0);
      ca = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, qa),
                                                   __builtin_bit_cast(bf16x8, la), ca, 0, 0, 0);
    }
    uint32_t up[4];
    uint32_t best = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t n = u * DSP_UNIT + 4 * kq + i;
      const float x = x0[i], d = err * ca[i] + tiny;
      const float slack = d + rnd * (__builtin_fabsf(c[i]) + d) +
                          ulp * (__builtin_fabsf(x) + __builtin_fabsf(c[i]));
      uint32_t lo, hi;
      if (!(ca[i] < 1e37f)) {
        lo = DSP_BOTTOM, hi = 0xffffffffu;  // an infinite or NaN operand: anything
      } else if (!(__builtin_fabsf(x) <= 3.40282346638528859812e38f)) {
        lo = ord_key(x);  // the bias is finite: NaN and -inf stay at the bottom, +inf at the top
        hi = lo == DSP_BOTTOM ? lo : 0xffffffffu;
      } else {
        lo = ord_key(x + c[i] - 2.f * slack);
        hi = ord_key(x + c[i] + 2.f * slack);
        // a bias below a quarter ulp of the logit leaves it as it is (logits masked with a large
        // negative value): the score is known
        if (__builtin_fabsf(c[i]) + d < __builtin_fabsf(x) * 1.4901161193847656e-08f && col < B &&
            n < a.v) {
          const uint64_t key = argmax_key(x, (uint32_t)n);
          known = key > known ? key : known;
          lo = hi = ord_key(x);
          if (lo > best) best = lo;
          hi = 0u;  // no candidate
        }
      }
      const bool live = col < B && n < a.v;
      up[i] = live ? hi : 0u;
      best = live && lo > best ? lo : best;
    }
    // the unit's largest lower bound of this lane's request (four lanes hold its rows)
    uint32_t o = (uint32_t)__shfl_xor((int)best, 16, WAVE);
    best = o > best ? o : best;
    o = (uint32_t)__shfl_xor((int)best, 32, WAVE);
    best = o > best ? o : best;
    low = best > low ? best : low;
    bool full = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (up[i] >= low && up[i] > DSP_BOTTOM) {
        const uint32_t at = atomicAdd(&s_n, 1u);
        full |= at >= DSP_CAND;
        if (at < DSP_CAND) {
          s_up[at] = up[i];
          s_row[at] = (uint32_t)(u * DSP_UNIT + 4 * kq + i);
          s_req[at] = (uint8_t)col;
        }
      }
    }
    if (__ballot(full)) break;  // the exact sums of every row follow
#pragma unroll
    for (int s = 0; s < KS; ++s) q0[s] = q1[s];
#pragma unroll
    for (int i = 0; i < 4; ++i) x0[i] = x1[i];
  }
  if (lane < B) atomicMax(&s_low[lane], low);
  if (known) atomicMax((unsigned long long*)&s_best[col], (unsigned long long)known);
  __syncthreads();
  // the exact scores of the candidates that the workgroup's lower bounds leave
  auto best_of = [&](int r, uint64_t key) {
    if (key > s_best[r]) atomicMax((unsigned long long*)&s_best[r], (unsigned long long)key);
  };
  auto by_wave = [&](int c) {  // one candidate by a wave: one round trip to memory
    const int r = s_req[c];
    const uint64_t key = dsp_exact_key(a, s_lat + r * R, r, s_row[c]);
    if (lane == 0) best_of(r, key);
  };
  const int n = (int)s_n;  // (uniform, as every branch on it)
  if (n <= DSP_FEW) {
    for (int c = w; c < n; c += DSP_WAVES)
      if (s_up[c] >= s_low[s_req[c]]) by_wave(c);
  } else if (n <= DSP_CAND) {
    for (int c = t; c < n; c += DSP_NT)
      if (s_up[c] >= s_low[s_req[c]]) s_left[atomicAdd(&s_m, 1u)] = (uint16_t)c;
    __syncthreads();
    const int m = (int)s_m;
    if (m <= DSP_FEW / 2) {
      for (int i = w; i < m; i += DSP_WAVES) by_wave(s_left[i]);
    } else {  // near ties (equal scores): a lane each
      for (int i = w * WAVE; i < m; i += DSP_NT) {
        const int c = s_left[i + lane < m ? i + lane : m - 1], r = s_req[c];
        uint64_t key[1];
        dsp_lane_keys<1>(a, s_lat, r, s_row[c], key);
        best_of(r, key[0]);
      }
    }
  } else {
    // more than the workgroup keeps (equal scores, several requests): every row, a lane each
    const int64_t tiles = (a.v + WAVE - 1) / WAVE;
    const int own = (int)((tiles - blockIdx.x + G - 1) / G);
    constexpr int NR = 4;
    const int parts = (B + NR - 1) / NR;
    for (int p = w; p < own * parts; p += DSP_WAVES) {
      const int r0 = p % parts * NR;
      const int64_t row = (blockIdx.x + (int64_t)(p / parts) * G) * WAVE + lane;
      uint64_t key[NR];
      dsp_lane_keys<NR>(a, s_lat, r0, row < a.v ? row : a.v - 1, key);
#pragma unroll
      for (int i = 0; i < NR; ++i)
        if (r0 + i < B) best_of(r0 + i, key[i]);
    }
  }
  __syncthreads();
  uint64_t* wg_keys = a.partial;                          // [b][G]
  uint64_t* group_keys = a.partial + (int64_t)B * G;      // [b][groups]
  if (t < B) {
    __hip_atomic_store(&wg_keys[(int64_t)t * G + blockIdx.x], s_best[t], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  const int group = blockIdx.x / DSP_GROUP, groups = (G + DSP_GROUP - 1) / DSP_GROUP;
  const int g0 = group * DSP_GROUP, gn = G - g0 < DSP_GROUP ? G - g0 : DSP_GROUP;
  if (!dsp_arrive(&g_dsp_group[group], gn, blockIdx.x == g0, &s_flag)) return;
  // the group's last workgroup: its group's keys, one load per lane
  for (int r = w; r < B; r += DSP_WAVES) {
    uint64_t m = lane < gn ? dsp_load(&wg_keys[(int64_t)r * G + g0 + lane]) : 0;
    m = wave_max_u64(m);
    if (lane == 0)
      __hip_atomic_store(&group_keys[r * groups + group], m, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!dsp_arrive(&g_dsp_cnt, groups, group == 0, &s_flag)) return;
  // the last group: the pick, one wave per request
  for (int r = w; r < B; r += DSP_WAVES) {
    uint64_t m = lane < groups ? dsp_load(&group_keys[r * groups + lane]) : 0;
    m = wave_max_u64(m);
    const int64_t at = (int64_t)r * a.block + j;
    if (lane == 0) a.out[at] = (int64_t)argmax_key_index(m);
  }
}

int64_t dsp_nwg(int64_t v) {
  const int64_t tiles = (v + WAVE - 1) / WAVE;
  const int64_t g = (tiles + DSP_WAVES - 1) / DSP_WAVES;
  return g < DSP_GRID ? g : DSP_GRID;
}

// Workgroups of a launch: as many as the registers of the rank's kernel let reside together.
int dsp_launch(int64_t v, int64_t rank) {
  const int64_t g = dsp_nwg(v), most = rank <= 128 ? DSP_GRID : 512;
  return g < most ? (int)g : (int)most;
}

}  // namespace

// Bytes of a packed [n, k] bf16 weight: the same as the source, so the reference can view the
// buffer as [n, k] (snowllm/ops/dspark.py:11-14). k % 8 == 0.
SV_API int64_t snowllm_dspark_weight_bytes(int64_t n, int64_t k) {
  if (n <= 0 || k <= 0 || k % 8) return 0;
  return n * k * 2;
}

SV_API int snowllm_dspark_pack_weight(const void* raw, void* packed, int64_t n, int64_t k,
                                      void* stream) {
  if (!raw || !packed || n <= 0 || k <= 0 || k % 8 || raw == packed) return SV_EINVAL;
  const int64_t chunks = n * (k / 8);
  hipLaunchKernelGGL(dsp_pack_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const uint16_t*)raw, (uint16_t*)packed, n, k);
  SV_CHECK_LAUNCH();
  return SV_OK;
}

// Workspace of snowllm_dspark_markov: 8-byte keys per request for every workgroup and
// every group of workgroups.
SV_API int64_t snowllm_dspark_markov_workspace_bytes(int64_t b, int64_t v, int64_t rank,
                                                     int64_t block) {
  (void)rank;
  (void)block;
  if (b <= 0 || v <= 0) return 0;
  const int64_t g = dsp_nwg(v);
  return ((b * (g + (g + DSP_GROUP - 1) / DSP_GROUP) * 8 + 255) / 256) * 256;
}

// base f32 [b * block, >= v] (row stride base_stride), w1 bf16 [v, rank], w2 packed by
// snowllm_dspark_pack_weight, anchor i64 [b] -> out i64 [b, block]; with confidence (f32
// [b, block]) also pre_head bf16 [b * block, >= h] (row stride ps), conf_weight f32
// [h + rank] and an optional scalar conf_bias. fp32_bias keeps the bias in fp32 instead of
// bf16. b <= 16, rank % 8 == 0, rank <= 512, b rank <= 4096. Calls on one device must be
// stream-ordered.
SV_API int snowllm_dspark_markov(const void* base, const void* w1, const void* w2,
                                 const int64_t* anchor, const void* pre_head,
                                 const float* conf_weight, const float* conf_bias, int64_t* out,
                                 float* confidence, void* workspace, int64_t b, int64_t v,
                                 int64_t rank, int64_t block, int64_t base_stride, int64_t h,
                                 int64_t ps, int64_t workspace_bytes, int fp32_bias,
                                 void* stream) {
  if (!base || !w1 || !w2 || !anchor || !out || !workspace) return SV_EINVAL;
  if (b <= 0 || b > DSP_MAX_B || v <= 0 || v > DSP_MAX_V || rank <= 0 || rank % 8 ||
      rank > DSP_MAX_RANK || b * rank > 4096 || block <= 0 || block > 1024 || base_stride < v)
    return SV_EINVAL;
  if (confidence && (!pre_head || !conf_weight || h <= 0 || ps < h)) return SV_EINVAL;
  if (workspace_bytes < snowllm_dspark_markov_workspace_bytes(b, v, rank, block)) return SV_EINVAL;
  DspArgs a{(const float*)base, (const uint16_t*)w1, (const uint16_t*)w2, anchor,
            (const uint16_t*)pre_head, conf_weight, conf_bias, out, confidence,
            (uint64_t*)workspace, v, base_stride, ps, (int)b, (int)rank, (int)block,
            confidence ? (int)h : 0, dsp_launch(v, rank), fp32_bias != 0, 0};
  for (int j = 0; j < block; ++j) {
    a.j = j;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(a.nwg + (confidence ? 1 : 0))), dim3(DSP_NT), 0,
                         (hipStream_t)stream, a);
    };
    if (rank <= 64) go(dsp_markov_kernel<2>);
    else if (rank <= 128) go(dsp_markov_kernel<4>);
    else if (rank <= 256) go(dsp_markov_kernel<8>);
    else go(dsp_markov_kernel<16>);
    SV_CHECK_LAUNCH();
  }
  return SV_OK;
}
