// Flash attention in float32 arithmetic on CDNA4 matrix cores (v_mfma_f32_32x32x2f32): float32,
// f16 and bf16 storage, head dims up to 128 in multiples of 4 (hd and hd_v may differ), any scale,
// rectangular keys, causal and key masks. Scores, probabilities and dS stay float32 throughout, as
// in the general-width kernels (sdpa_rows.hip) this takes calls over from.
//
// What bounds it: the float32 matrix rate (157 TFLOP/s; a 32x32x2 product takes its SIMD 64 cycles),
// and beside it every vector instruction: measured, a wave's or its neighbours' VALU work does not run
// under a float32 product (65 cycles a product alone, 130 with 16 multiply-adds between, at one or two
// waves a SIMD), as it does under a 16-bit one. So a tile costs the sum of both, and the softmax
// arithmetic is kept short. Loads are cheap beside that: a wave takes its operand fragments straight
// from memory (L1 and L2) into registers, converted on the way, with no LDS tile and no barrier in the
// loop (fetching them a tile ahead changed nothing). The orientation is the 16-bit family's
// (sdpa_mfma.h): the resident rows are the N side, a lane owns one resident row (n = lane % 32, shared
// with lane ^ 32), and an accumulator item of the score tile *is* the B operand of one step of the next
// product: item i of half h = lane / 32 covers streamed row 8 (i / 4) + 4 h + i % 4, so step i
// multiplies those two rows, and no value changes lanes between the products.
//   forward:  S^T = K Q^T                   then  O^T  += V^T P^T
//   dQ pass:  S^T = K Q^T, dP^T = V dO^T,   dQ^T += K^T dS^T
//   dKV pass: S = Q K^T, dP = dO V^T,       dV^T += dO^T P,  dK^T += Q^T dS
//
// A workgroup is four waves. KS = 4: one 32-row block, the waves taking streamed tiles w, w + 4, ...
// and their totals combined at the end through LDS in wave order. KS = 1: four blocks, a wave each,
// from 8192 blocks on or where few tiles stream (WIDE_WAVES, WIDE_SHORT). Every total is formed in a fixed order.
//
// Measured, us, rows kernels -> these (forward, dQ, dK/dV), float32 causal: 48 heads x 1024 rows x 32
// dims 756, 912, 1140 -> 48, 60, 90; 8 x 256 x 64 22, 23, 38 -> 12, 15, 19; 64 x 512 x 64 329, 390, 500
// -> 40, 56, 88 (paired blocks; unpaired 57, 71, 100); 16 x 2048 x 64, full, 1252, 1531, 2125 -> 178,
// 246, 421 (90 TFLOP/s); f16, 256 heads, 197 x 1021 x 80, key mask, dQ and dK/dV 3765, 2552 -> 480, 692.
//
// Accuracy: a tile's product starts from zero and is added to the running total once per tile (with
// the forward's rescale, one fused operation), so a total over thousands of rows is a sum of
// 32-row sums; exponentials are within 2 ulp (wide_exp).

#pragma once

#include "sdpa.h"

namespace limn {
namespace {

constexpr int WT = 32;          // rows per tile, resident and streamed
constexpr int WTHREADS = 256;
constexpr int FAR = 0x7f000000;  // a byte offset past every matrix: its load reads zero

__device__ __forceinline__ float wide_inf() { return __builtin_inff(); }

__device__ __forceinline__ f32x16 wide_zero() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; i++) z[i] = 0.f;
  return z;
}

// x combined with the other lane of its row (lane ^ 32)
__device__ __forceinline__ float wide_pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wide_pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// e^x within 2 ulp of float: the hardware's 2^t at t = x log2(e) rounded, times 1 + ln 2 times what t
// lost to that rounding (an fma recovers it, and log2(e)'s own tail adds the rest). Six operations
// against some fifteen of expf; a row's exponentials run beside its products on the same SIMD. Far
// below zero it is 0 (where -inf, a hidden key's score, must not meet itself in the fma); NaN stays.
__device__ __forceinline__ float wide_exp(float x) {
  constexpr float LOG2E = 0x1.715476p+0f, TAIL = 0x1.4ae0cp-26f, LN2 = 0x1.62e43p-1f;
  x = x < -200.f ? -200.f : x;
  const float t = x * LOG2E;
  const float lost = fmaf(x, TAIL, fmaf(x, LOG2E, -t));
  return fast_exp2(t) * fmaf(lost, LN2, 1.f);
}

// s scale - L with the product rounded first, as in L itself: a row that one key dominates then has weight
// 1, not e^(what the rounding of a far score took). At scores 64 times the usual spread dV was 5.0e-6 off
// float64 without, 2.9e-6 with.
__device__ __forceinline__ float wide_logit(float s, float scale, float L) {
#pragma clang fp contract(off)
  return s * scale - L;
}

template <typename T>
__device__ __forceinline__ f32x4 wide_load4(__amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (sizeof(typename T::Storage) == 4) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  } else {
    const u16x4 v = __builtin_bit_cast(u16x4, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    return f32x4{T::unpack(v[0]), T::unpack(v[1]), T::unpack(v[2]), T::unpack(v[3])};
  }
}
template <typename T>
__device__ __forceinline__ float wide_load1(__amdgpu_buffer_rsrc_t r, int off, int scalar = 0) {
  if constexpr (sizeof(typename T::Storage) == 4)
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, scalar, 0));
  else
    return T::unpack(__builtin_amdgcn_raw_buffer_load_b16(r, off, scalar, 0));
}

// One head's (rows x width) matrix, width <= D a multiple of 4. Rows past the end and dims past the
// width read as zeros: the buffer ends with the matrix, and a lane whose dims do not exist reads
// from FAR.
template <typename T, int D>
struct WideRows {
  static constexpr int SZ = sizeof(typename T::Storage);
  __amdgpu_buffer_rsrc_t rsrc;
  int rb, width;  // bytes of a row; dims
  __device__ __forceinline__ WideRows(const typename T::Storage* base, int rows, int width_) {
    width = width_;
    rb = width_ * SZ;
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, rows * rb, 0x00020000);
  }
  // row operand: out[g] = dims 8 g + 4 h .. + 3 of row row0 + n
  __device__ __forceinline__ void rows(int row0, f32x4 (&out)[D / 8]) const {
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    const int at = (row0 + n) * rb + 4 * h * SZ;
#pragma unroll
    for (int g = 0; g < D / 8; g++) out[g] = wide_load4<T>(rsrc, 8 * g + 4 * h < width ? at + 8 * g * SZ : FAR);
  }
  // transposed operand of dims 32 dt .. + 31: out[i] = dim 32 dt + n of row row0 + 8 (i / 4) + 4 h + i % 4.
  // The item's row is a scalar offset, which the range check subtracts from the buffer's size: a
  // matrix has at least 32 rows (wide_takes), so that stays positive.
  __device__ __forceinline__ void columns(int row0, int dt, float (&out)[16]) const {
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    const int d = dt * 32 + n, at = d < width ? (row0 + 4 * h) * rb + d * SZ : FAR;
#pragma unroll
    for (int i = 0; i < 16; i++) out[i] = wide_load1<T>(rsrc, at, (8 * (i >> 2) + (i & 3)) * rb);
  }
  // one element of row `row`
  __device__ __forceinline__ float at(int row, int d) const { return wide_load1<T>(rsrc, d < width ? row * rb + d * SZ : FAR, 0); }
};

// the product of two row operands over all D dims: SPAN dims at a time in chains that start from zero,
// two chains, or one past 64 dims, where the registers of a second one spill (128 dims, 32 heads x 1024
// rows, dK/dV: 494 us with two, 269 with two chains over all dims).
template <int D, int SPAN>
__device__ __forceinline__ f32x16 wide_dots(const f32x4 (&a)[D / 8], const f32x4 (&b)[D / 8]) {
  f32x16 s;
#pragma unroll
  for (int g0 = 0; g0 < D / 8; g0 += SPAN / 8) {
    f32x16 c0 = wide_zero(), c1 = wide_zero();
#pragma unroll
    for (int g = g0; g < g0 + SPAN / 8; g++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (D > 64 || j % 2 == 0) c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g][j], b[g][j], c0, 0, 0, 0);
        else c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g][j], b[g][j], c1, 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float c = D > 64 ? c0[i] : c0[i] + c1[i];
      s[i] = g0 == 0 ? c : s[i] + c;
    }
  }
  return s;
}

// Scores: their error counts in full in the exponential (and a row's sum of weights), so their chains are
// as short as the rows kernels' quarter rows: 8 products at 32 dims, 16 past that. With twice that, outputs
// of 24 heads x 512 rows x 32 dims, causal, were 1.46e-7 off float64 against the rows kernels' 1.37e-7, now
// 1.36e-7; 96 dims 1.71e-7 against 1.55e-7, now 1.53e-7. It costs 0-4%.
template <int D>
__device__ __forceinline__ f32x16 wide_scores(const f32x4 (&a)[D / 8], const f32x4 (&b)[D / 8]) {
  return wide_dots<D, D == 64 ? 32 : 16>(a, b);
}

// the 32-row sum of columns x probabilities, in two chains
__device__ __forceinline__ f32x16 wide_mix(const float (&a)[16], const f32x16& p) {
  f32x16 c0 = wide_zero(), c1 = wide_zero();
#pragma unroll
  for (int i = 0; i < 8; i++) {
    c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], p[i], c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i + 8], p[i + 8], c1, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 16; i++) c0[i] += c1[i];
  return c0;
}

__device__ __forceinline__ bool wide_bad(float x) { return __builtin_amdgcn_classf(x, 0x207); }  // NaN or infinite

// Columns of a tile some of whose pairs are no term of the sum (right of the diagonal, masked, past the
// end): their weight is zero, but zero times a NaN or an infinity in such a row is not. Clears every
// non-finite value; whether there was one.
__device__ __forceinline__ bool wide_clean(float (&a)[16]) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    bad |= wide_bad(a[i]);
    a[i] = wide_bad(a[i]) ? 0.f : a[i];
  }
  return __any(bad);
}

// The non-finite terms that wide_clean took out and that do belong to lane n's sum: `terms` bit r is
// set when streamed row row0 + r does. The rare path of an already broken input.
template <typename T, int D>
__device__ __forceinline__ f32x16 wide_amend(f32x16 o, const WideRows<T, D>& m, int row0, int dt, const f32x16& p, unsigned terms) {
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
#pragma unroll 1
  for (int r = 0; r < WT; r++) {
    const int item = 4 * (r >> 3) + (r & 3), half = (r >> 2) & 1;
    float w = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) w = i == item ? p[i] : w;
    w = __shfl(w, n + 32 * half);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float x = m.at(row0 + r, dt * 32 + 8 * (i >> 2) + 4 * h + (i & 3));
      o[i] = wide_bad(x) && ((terms >> r) & 1u) ? fmaf(w, x, o[i]) : o[i];
    }
  }
  return o;
}

// wide_mix of columns (row0, dt) of m; `edge` (uniform) when not every pair is a term
template <typename T, int D>
__device__ __forceinline__ f32x16 wide_mix_tile(const WideRows<T, D>& m, float (&a)[16], int row0, int dt, const f32x16& p, bool edge, unsigned terms) {
  bool bad = false;
  if (edge) bad = wide_clean(a);
  const f32x16 o = wide_mix(a, p);
  return bad ? wide_amend<T, D>(o, m, row0, dt, p, terms) : o;
}

// lane n's row of an accumulator set, dims 32 dt + 8 g + 4 h .. + 3 in items 4 g ..
template <typename T, int D>
__device__ __forceinline__ void wide_store(typename T::Storage* base, const f32x16 (&acc)[D / 32], int row, int rows, int width,
                                           float mul) {
  if (row >= rows) return;
  const int h = (threadIdx.x >> 5) & 1;
  typename T::Storage* o = base + (int64_t)row * width;
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int d = dt * 32 + 8 * g + 4 * h;
      if (d < width) {
#pragma unroll
        for (int e = 0; e < 4; e++) T::store(o, d + e, acc[dt][4 * g + e] * mul);
      }
    }
}

// The four waves' accumulators added into wave 0's, in wave order. `space` holds 3 images of
// 64 lanes x D / 2 values.
template <int D>
__device__ __forceinline__ void wide_combine(f32x16 (&acc)[D / 32], float* space, int wave) {
  const int lane = threadIdx.x & 63;
  if (wave > 0) {
    float* mine = space + (wave - 1) * 64 * (D / 2) + lane;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int i = 0; i < 16; i++) mine[(dt * 16 + i) * 64] = acc[dt][i];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 0; w < 3; w++)
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[dt][i] += space[(w * (D / 2) + dt * 16 + i) * 64 + lane];
  }
}

// Which head and unit of blocks a wave works on. Workgroup id runs on XCD id % 8: each XCD takes a
// contiguous run of heads, so that a head's streamed matrix stays in one L2. A unit is a block (KS =
// 4) or four (KS = 1), or with `pair` (KS = 4, causal) a block and its mirror, the block counted from
// the other end: every workgroup then walks the same number of tiles, in one round.
template <int KS>
__device__ __forceinline__ int wide_units(int blocks, int pair) {
  return KS == 1 ? (blocks + 3) / 4 : pair ? (blocks + 1) / 2 : blocks;
}
template <int KS>
__device__ __forceinline__ void wide_place(int blocks, int pair, int64_t& b, int& unit) {
  const int units = wide_units<KS>(blocks, pair);
  int64_t id = blockIdx.x;
  if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
  b = id / units;
  unit = (int)(id - b * units);
}

// the live keys of a tile as one word: bit r = key k0 + r exists and is not masked
template <typename T>
__device__ __forceinline__ unsigned wide_live(__amdgpu_buffer_rsrc_t mask, bool masked, int k0, int t_k) {
  const int n = threadIdx.x & 31;
  bool live = k0 + n < t_k;
  if (masked) live = live && wide_load1<T>(mask, (k0 + n) * (int)sizeof(typename T::Storage)) != 0.f;
  return (unsigned)__ballot(live);
}

template <typename T, int D, int KS>
__global__ __launch_bounds__(WTHREADS, D <= 32 ? 4 : 2) void sdpa_fwd_wide(
    const typename T::Storage* __restrict__ q, const typename T::Storage* __restrict__ k, const typename T::Storage* __restrict__ v,
    const typename T::Storage* __restrict__ mask, typename T::Storage* __restrict__ out, float* __restrict__ lse, int64_t batch,
    int t_q, int t_k, int hd, int hd_v, int causal, int pair, float scale) {
  constexpr int SZ = sizeof(typename T::Storage);
  __shared__ float space[KS == 1 ? 1 : 3 * 64 * (D / 2)];
  __shared__ float stat[KS == 1 ? 1 : 2 * 4 * 64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, n = lane & 31;
  const int blocks = (t_q + WT - 1) / WT;
  int64_t b;
  int unit;
  wide_place<KS>(blocks, pair, b, unit);
  const int reps = pair && blocks - 1 - unit != unit ? 2 : 1;
#pragma unroll 1
  for (int rep = 0; rep < reps; rep++) {
  // causal: the longest rows go first
  const int blk = blocks - 1 - (KS == 1 ? unit * 4 + wave : rep == 0 ? unit : blocks - 1 - unit);
  if (KS == 1 && blk < 0) return;  // no barrier follows
  const int q0 = blk * WT, row = q0 + n;
  const WideRows<T, D> qm(q + b * (int64_t)t_q * hd, t_q, hd), km(k + b * (int64_t)t_k * hd, t_k, hd), vm(v + b * (int64_t)t_k * hd_v, t_k, hd_v);
  const __amdgpu_buffer_rsrc_t mm = __builtin_amdgcn_make_buffer_rsrc((void*)(mask + (mask != nullptr ? b * (int64_t)t_k : 0)), (short)0, mask != nullptr ? t_k * SZ : 0, 0x00020000);

  f32x4 qf[D / 8];
  qm.rows(q0, qf);
  f32x16 acc[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++) acc[dt] = wide_zero();
  float m = -wide_inf(), l = 0.f;
  const int kend = causal && q0 + WT < t_k ? q0 + WT : t_k;
  for (int k0 = (KS == 1 ? 0 : wave * WT); k0 < kend; k0 += KS * WT) {
    f32x4 kf[D / 8];
    km.rows(k0, kf);
    const unsigned live = wide_live<T>(mm, mask != nullptr, k0, t_k);
    f32x16 s = wide_scores<D>(kf, qf);
    const bool edge = live != ~0u || (causal && k0 + WT - 1 > q0);
    unsigned terms = live;
    if (edge) {
      if (causal) terms &= row - k0 >= 31 ? ~0u : row < k0 ? 0u : (2u << (row - k0)) - 1u;
#pragma unroll
      for (int i = 0; i < 16; i++) s[i] = (terms >> (8 * (i >> 2) + 4 * h + (i & 3))) & 1u ? s[i] * scale : -wide_inf();
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++) s[i] *= scale;
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, s[i]);
    mx = fmaxf(m, wide_pair_max(mx));
    const float base = mx == -wide_inf() ? 0.f : mx;
    const float alpha = wide_exp(m - base);  // m = -inf: 0
    m = mx;
    float rs = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      s[i] = wide_exp(s[i] - base);
      rs += s[i];
    }
    l = fmaf(l, alpha, rs);
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++) {
      float vc[16];
      vm.columns(k0, dt, vc);
      const f32x16 o = wide_mix_tile<T, D>(vm, vc, k0, dt, s, edge, terms);
#pragma unroll
      for (int i = 0; i < 16; i++) acc[dt][i] = fmaf(acc[dt][i], alpha, o[i]);
    }
  }
  if constexpr (KS > 1) {
    stat[wave * 64 + lane] = m;
    __syncthreads();
    float mr = stat[lane];
#pragma unroll
    for (int w = 1; w < 4; w++) mr = fmaxf(mr, stat[w * 64 + lane]);
    const float f = m == -wide_inf() ? 0.f : wide_exp(m - mr);
    stat[256 + wave * 64 + lane] = l * f;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[dt][i] *= f;
    wide_combine<D>(acc, space, wave);  // its barrier also covers the sums of `stat`
    m = mr;
    l = ((stat[256 + lane] + stat[320 + lane]) + stat[384 + lane]) + stat[448 + lane];
  }
  if (KS == 1 || wave == 0) {
    const float total = wide_pair_sum(l);
    wide_store<T, D>(out + b * (int64_t)t_q * hd_v, acc, row, t_q, hd_v, 1.f / total);
    if (h == 0 && row < t_q) lse[b * (int64_t)t_q + row] = m + logf(total);
  }
  if (KS > 1) __syncthreads();  // the pair's second block reuses the LDS arrays
  }
}

template <typename T, int D, int KS>
__global__ __launch_bounds__(WTHREADS, D <= 32 ? 3 : D <= 64 ? 2 : 1) void sdpa_bwd_q_wide(
    const typename T::Storage* __restrict__ q, const typename T::Storage* __restrict__ k, const typename T::Storage* __restrict__ v,
    const typename T::Storage* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    const typename T::Storage* __restrict__ mask, typename T::Storage* __restrict__ dq, int64_t batch, int t_q, int t_k, int hd,
    int hd_v, int causal, int pair, float scale) {
  constexpr int SZ = sizeof(typename T::Storage);
  __shared__ float space[KS == 1 ? 1 : 3 * 64 * (D / 2)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, n = lane & 31;
  const int blocks = (t_q + WT - 1) / WT;
  int64_t b;
  int unit;
  wide_place<KS>(blocks, pair, b, unit);
  const int reps = pair && blocks - 1 - unit != unit ? 2 : 1;
#pragma unroll 1
  for (int rep = 0; rep < reps; rep++) {
  // causal: the longest rows go first
  const int blk = blocks - 1 - (KS == 1 ? unit * 4 + wave : rep == 0 ? unit : blocks - 1 - unit);
  if (KS == 1 && blk < 0) return;  // no barrier follows
  const int q0 = blk * WT, row = q0 + n;
  const WideRows<T, D> qm(q + b * (int64_t)t_q * hd, t_q, hd), om(dout + b * (int64_t)t_q * hd_v, t_q, hd_v);
  const WideRows<T, D> km(k + b * (int64_t)t_k * hd, t_k, hd), vm(v + b * (int64_t)t_k * hd_v, t_k, hd_v);
  const __amdgpu_buffer_rsrc_t mm = __builtin_amdgcn_make_buffer_rsrc((void*)(mask + (mask != nullptr ? b * (int64_t)t_k : 0)), (short)0, mask != nullptr ? t_k * SZ : 0, 0x00020000);

  f32x4 qf[D / 8], of[D / 8];
  qm.rows(q0, qf);
  om.rows(q0, of);
  f32x16 acc[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++) acc[dt] = wide_zero();
  const float L = row < t_q ? lse[b * (int64_t)t_q + row] : 0.f, Dr = row < t_q ? delta[b * (int64_t)t_q + row] : 0.f;
  const int kend = causal && q0 + WT < t_k ? q0 + WT : t_k;
  for (int k0 = (KS == 1 ? 0 : wave * WT); k0 < kend; k0 += KS * WT) {
    f32x4 kf[D / 8], vf[D / 8];
    km.rows(k0, kf);
    vm.rows(k0, vf);
    const unsigned live = wide_live<T>(mm, mask != nullptr, k0, t_k);
    f32x16 s = wide_scores<D>(kf, qf);
    const f32x16 dp = wide_dots<D, 32>(vf, of);
    // a key that exists but is hidden has probability exp(-inf - L): zero, or NaN in a row whose
    // every key is hidden (L = -inf), as the numpy reference's; one past t_k or right of the row
    // is no term of the sum at all
    const bool edge = live != ~0u || (causal && k0 + WT - 1 > q0);
    unsigned terms = live;
    if (edge) {
      const int last = (causal && row < t_k ? row : t_k - 1) - k0;
      const unsigned present = last >= 31 ? ~0u : last < 0 ? 0u : (2u << last) - 1u;
      terms &= present;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int r = 8 * (i >> 2) + 4 * h + (i & 3);
        const float x = wide_exp(((live >> r) & 1u ? s[i] * scale : -wide_inf()) - L);
        s[i] = (terms >> r) & 1u ? x * (dp[i] - Dr) * scale : (present >> r) & 1u ? x : 0.f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++) s[i] = wide_exp(fmaf(s[i], scale, -L)) * (dp[i] - Dr) * scale;
    }
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++) {
      float kc[16];
      km.columns(k0, dt, kc);
      const f32x16 o = wide_mix_tile<T, D>(km, kc, k0, dt, s, edge, terms);
#pragma unroll
      for (int i = 0; i < 16; i++) acc[dt][i] += o[i];
    }
  }
  if constexpr (KS > 1) wide_combine<D>(acc, space, wave);
  if (KS == 1 || wave == 0) wide_store<T, D>(dq + b * (int64_t)t_q * hd, acc, row, t_q, hd, 1.f);
  if (KS > 1) __syncthreads();  // the pair's second block reuses the LDS array
  }
}

template <typename T, int D, int KS>
__global__ __launch_bounds__(WTHREADS, D <= 32 ? 2 : 1) void sdpa_bwd_kv_wide(
    const typename T::Storage* __restrict__ q, const typename T::Storage* __restrict__ k, const typename T::Storage* __restrict__ v,
    const typename T::Storage* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    const typename T::Storage* __restrict__ mask, typename T::Storage* __restrict__ dk, typename T::Storage* __restrict__ dv,
    int64_t batch, int t_q, int t_k, int hd, int hd_v, int causal, int pair, float scale) {
  __shared__ float space[KS == 1 ? 1 : 3 * 64 * (D / 2)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, n = lane & 31;
  const int blocks = (t_k + WT - 1) / WT;
  int64_t b;
  int unit;
  wide_place<KS>(blocks, pair, b, unit);
  const int reps = pair && blocks - 1 - unit != unit ? 2 : 1;
#pragma unroll 1
  for (int rep = 0; rep < reps; rep++) {
  // causal: the first keys are seen by the most queries, and go first
  const int blk = KS == 1 ? unit * 4 + wave : rep == 0 ? unit : blocks - 1 - unit;
  if (KS == 1 && blk >= blocks) return;  // no barrier follows
  const int k0 = blk * WT, key = k0 + n;
  const WideRows<T, D> qm(q + b * (int64_t)t_q * hd, t_q, hd), om(dout + b * (int64_t)t_q * hd_v, t_q, hd_v);
  const WideRows<T, D> km(k + b * (int64_t)t_k * hd, t_k, hd), vm(v + b * (int64_t)t_k * hd_v, t_k, hd_v);
  const __amdgpu_buffer_rsrc_t lm = __builtin_amdgcn_make_buffer_rsrc((void*)(lse + b * (int64_t)t_q), (short)0, t_q * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t dm = __builtin_amdgcn_make_buffer_rsrc((void*)(delta + b * (int64_t)t_q), (short)0, t_q * 4, 0x00020000);

  f32x4 kf[D / 8], vf[D / 8];
  km.rows(k0, kf);
  vm.rows(k0, vf);
  const bool live = mask == nullptr || key >= t_k || T::load(mask, b * (int64_t)t_k + key) != 0.f;
  const bool dead = __any(!live);  // a hidden key in the block: every tile takes the edge form
  f32x16 gk[D / 32], gv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++) {
    gk[dt] = wide_zero();
    gv[dt] = wide_zero();
  }
  for (int r0 = (causal ? k0 : 0) + (KS == 1 ? 0 : wave * WT); r0 < t_q; r0 += KS * WT) {
    f32x4 qf[D / 8], of[D / 8], l4[4], d4[4];
    qm.rows(r0, qf);
    om.rows(r0, of);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      l4[g] = wide_load4<F32>(lm, (r0 + 8 * g + 4 * h) * 4);
      d4[g] = wide_load4<F32>(dm, (r0 + 8 * g + 4 * h) * 4);
    }
    f32x16 p = wide_scores<D>(qf, kf);
    f32x16 ds = wide_dots<D, D == 128 ? 16 : 32>(of, vf);  // at 128 dims the longer span spills: 16 x 2048 rows 1037 us, 897
    const bool edge = dead || r0 + WT > t_q || (causal && r0 < k0 + WT - 1);
    unsigned terms = ~0u;
    if (edge) {
      const int from = causal ? key - r0 : 0, past = t_q - r0;  // this key's queries of the tile: [from, past)
      terms = (from <= 0 ? ~0u : from > 31 ? 0u : ~0u << from) & (past > 31 ? ~0u : (1u << past) - 1u);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int r = 8 * (i >> 2) + 4 * h + (i & 3);
        const bool term = (terms >> r) & 1u;
        const float x = wide_exp((live ? p[i] * scale : -wide_inf()) - l4[i >> 2][i & 3]);
        p[i] = term ? x : 0.f;
        ds[i] = term ? x * (ds[i] - d4[i >> 2][i & 3]) * scale : 0.f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        p[i] = wide_exp(wide_logit(p[i], scale, l4[i >> 2][i & 3]));
        ds[i] = p[i] * (ds[i] - d4[i >> 2][i & 3]) * scale;
      }
    }
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++) {
      float c[16];
      om.columns(r0, dt, c);
      f32x16 o = wide_mix_tile<T, D>(om, c, r0, dt, p, edge, terms);
#pragma unroll
      for (int i = 0; i < 16; i++) gv[dt][i] += o[i];
      qm.columns(r0, dt, c);
      o = wide_mix_tile<T, D>(qm, c, r0, dt, ds, edge, terms);
#pragma unroll
      for (int i = 0; i < 16; i++) gk[dt][i] += o[i];
    }
  }
  if constexpr (KS > 1) {
    wide_combine<D>(gk, space, wave);
    __syncthreads();  // wave 0 has read every image before the next ones land
    wide_combine<D>(gv, space, wave);
  }
  if (KS == 1 || wave == 0) {
    wide_store<T, D>(dk + b * (int64_t)t_k * hd, gk, key, t_k, hd, 1.f);
    wide_store<T, D>(dv + b * (int64_t)t_k * hd_v, gv, key, t_k, hd_v, 1.f);
  }
  if (KS > 1) __syncthreads();  // the pair's second block reuses the LDS array
  }
}

template <typename T, int D, int KS>
int launch_wide(SdpaPass pass, const SdpaArgs& a) {
  typedef typename T::Storage S;
  const int64_t rows = pass == SDPA_BWD_KV ? a.t_k : a.t_q, blocks = (rows + WT - 1) / WT;
  const int pair = KS > 1 && a.causal && blocks >= 16 && a.batch * ((blocks + 1) / 2) >= WIDE_PAIRS;
  const int64_t groups = a.batch * (KS == 1 ? (blocks + 3) / 4 : pair ? (blocks + 1) / 2 : blocks);
  if (groups > 0x7fffffff) return fail(LIMN_HIP_EUNSUPPORTED, "sdpa: %lld workgroups exceed one launch", (long long)groups);
  const dim3 grid((unsigned)groups), block(WTHREADS);
  const int t_q = (int)a.t_q, t_k = (int)a.t_k, hd = (int)a.hd, hd_v = (int)a.hd_v, causal = a.causal ? 1 : 0;
  const float scale = (float)a.scale;
  const S *q = (const S*)a.q, *k = (const S*)a.k, *v = (const S*)a.v, *o = (const S*)a.dout, *m = (const S*)a.mask;
  const float *l = (const float*)a.lse, *d = (const float*)a.delta;
  if (pass == SDPA_FWD)
    hipLaunchKernelGGL((sdpa_fwd_wide<T, D, KS>), grid, block, 0, a.stream, q, k, v, m, (S*)a.out0, (float*)a.out1, a.batch, t_q,
                       t_k, hd, hd_v, causal, pair, scale);
  else if (pass == SDPA_BWD_Q)
    hipLaunchKernelGGL((sdpa_bwd_q_wide<T, D, KS>), grid, block, 0, a.stream, q, k, v, o, l, d, m, (S*)a.out0, a.batch, t_q, t_k,
                       hd, hd_v, causal, pair, scale);
  else
    hipLaunchKernelGGL((sdpa_bwd_kv_wide<T, D, KS>), grid, block, 0, a.stream, q, k, v, o, l, d, m, (S*)a.out0, (S*)a.out1,
                       a.batch, t_q, t_k, hd, hd_v, causal, pair, scale);
  return check_hip(hipGetLastError(), "launching an sdpa kernel");
}

template <typename T, int D>
int launch_wide_split(SdpaPass pass, const SdpaArgs& a) {
  const int64_t rows = pass == SDPA_BWD_KV ? a.t_k : a.t_q, streamed = pass == SDPA_BWD_KV ? a.t_q : a.t_k;
  const int64_t waves = a.batch * ((rows + WT - 1) / WT);
  const bool alone = waves >= WIDE_WAVES || streamed <= WT || (streamed <= 3 * WT && waves >= WIDE_SHORT);
  return alone ? launch_wide<T, D, 1>(pass, a) : launch_wide<T, D, 4>(pass, a);
}

// One storage type's instances (its own translation unit, so they compile in parallel).
template <typename T>
int launch_wide_type(SdpaPass pass, const SdpaArgs& a) {
  const int64_t width = a.hd > a.hd_v ? a.hd : a.hd_v;
  if (width <= 32) return launch_wide_split<T, 32>(pass, a);
  if (width <= 64) return launch_wide_split<T, 64>(pass, a);
  if (width <= 96) return launch_wide_split<T, 96>(pass, a);
  return launch_wide_split<T, 128>(pass, a);
}

}  // namespace
}  // namespace limn
