// Forward attention for f16 and bf16 at head dims the 16-bit family (sdpa_mfma.h) has no kernel for
// (any multiple of 8 up to 128, hd and hd_v may differ), without a causal mask: 16-bit matrix products
// with the float32 probabilities split into 16-bit parts.
//
// S = Q K^T has 16-bit operands as they are stored, so its products are exact either way. P is float32
// in the general-width kernels this takes calls over from; here it is a sum of 16-bit parts:
//   bf16: three, each the rounding of what the ones before it leave. They hold all 24 bits of P; two left
//     2^-19.5 of the terms' spread in an output whose terms cancel, where float32 leaves 2^-22.5.
//   f16: hi + 2^-12 lo, the lo products in totals of their own. 11 + 11 bits and a sign, so at most the last
//     bit of P is lost. f16 ends at 2^-24, so P carries a factor 2^SHIFT that its sum carries too: hi
//     reaches 2^15, the top of the range, when a row's reference point lags by its LAG, and so does lo. A
//     weight then loses at most 2^-49 of its row's largest (SHIFT + 12 + 25 bits down), a row less
//     than 2^-49 times its keys times the largest value, which f16 can show (2^-25) only past 2^24.
//     With no factor and hi and lo in one total a weight 2^-25 below the largest was dropped: a key of weight
//     1 and value 0 among 1020 others 17 nats below it left an output 20% off.
// Measured, us, two parts in one total / these: f16, 256 heads 197 x 1021 x 80, key mask, 57.0/57.3, 16 x 4096 x
// 4096 x 80 172/174, 64 x 1024 x 1024 x 120 60/64 (the second totals spill there); bf16 56.6/62.3, 166/198, 58/68.
//
// The structure is sdpa_fwd_mfma's: 128 queries a workgroup, 32 a wave, 64-key tiles staged through
// LDS a tile ahead, one lane per query row, the probability accumulators feeding the next product in
// place. Dims between the width and the padded D are zeros in the tile. What bounds it is the softmax
// arithmetic (exponentials, the split, the packing), which runs under the 16-bit products, as it does
// not under float32 ones.
//
// An infinity in a live V row reaches every query that gives its key weight, but a split weight with a part
// that is zero or negative would make it NaN. A workgroup with a NaN in its totals (from a value that is
// not finite, or a score that leaves float32) walks the keys once more with one small equal weight for
// each nonzero probability and no split, and stores what comes out non-finite: the sign of an infinity,
// NaN where infinities meet or the probability is 0 or NaN.

#include <type_traits>

#include "sdpa_mfma.h"

namespace limn {
namespace {

// Stage (sdpa_mfma.h) of K and V rows of their own widths, zero past them. V rows of keys that a key
// mask hides are cleared: their probability is zero, but zero times a NaN they may hold is not.
template <int D>
struct WidthStage {
  static constexpr int COLS = D / 8, PER_TILE = COLS * (TILE / 4), SLOTS = (2 * PER_TILE + THREADS - 1) / THREADS;
  u16x8 r[SLOTS][4];
  static_assert(PER_TILE % 64 == 0, "a wave's blocks come from one matrix");

  template <typename T, bool MASK>
  __device__ __forceinline__ void load(const Rows& k, const Rows& v, int hd, int hd_v, const MaskRow& mask, int row0) {
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
      const int idx = threadIdx.x + s * THREADS;
      if (idx < 2 * PER_TILE) {
        const int which = __builtin_amdgcn_readfirstlane(idx / PER_TILE), w = idx - which * PER_TILE;
        const int col = w % COLS, grp = w / COLS;
        const Rows& m = which ? v : k;
        const int width = which ? hd_v : hd;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int row = row0 + grp * 4 + e;
          r[s][e] = m.load8(col * 8 < width ? row * width + col * 8 : 0x3f000000);  // past the matrix: zeros
          if (MASK && which && T::unpack(mask.load(row)) == 0.f) r[s][e] = zero8();
        }
      }
    }
  }
  __device__ __forceinline__ void store(u16* tile0, u16* tile1) const {
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
      const int idx = threadIdx.x + s * THREADS;
      if (idx < 2 * PER_TILE) {
        const int which = idx / PER_TILE, w = idx - which * PER_TILE;
        u16* tile = which ? tile1 : tile0;
#pragma unroll
        for (int e = 0; e < 4; e++) *(u16x8*)(tile + tile_at<D>((w / COLS) * 4 + e, (w % COLS) * 8)) = r[s][e];
      }
    }
  }
};

// How a storage type splits P (see above): 16-bit parts, sets of totals, log2 of P's factor and how far
// (log2) a row's largest probability may pass its reference point.
template <typename T>
struct Split {  // bf16
  static constexpr int PARTS = 3, TOTALS = 1;
  static constexpr float SHIFT = 0.f, LAG = RESCALE_LOG2;
};
template <>
struct Split<F16> {
  static constexpr int PARTS = 2, TOTALS = 2;
  static constexpr float SHIFT = 12.f, LAG = 3.f;
};

// Reference points (log2 of a weight) past which the product of score and scale is off by more than 2^-5 of
// a power of two once rounded: the largest weight of a row would be 2^e times what it is, e growing with
// the score, and leave f16's range (from scores of 2^26 on) or float32's (2^31). The test for it is one
// comparison a tile: within 1% of the time without up to 96 dims, 64 -> 68 us in f16 at 64 x 1024 x 1024 x 120.
constexpr float FAR = 0x1p20f;

// Items base .. base + 7 of s as the parts of Split, most significant first.
template <typename T>
__device__ __forceinline__ void split8(const f32x16& s, int base, u16x8 (&part)[Split<T>::PARTS]) {
  part[0] = pack8<T>(s, base);
  if constexpr (Split<T>::TOTALS == 2) {
    const f16x8 hi = __builtin_bit_cast(f16x8, part[0]);
    f16x8 lo;
#pragma unroll
    for (int e = 0; e < 8; e++) lo[e] = (_Float16)fmaf((float)hi[e], -0x1p12f, s[base + e] * 0x1p12f);
    part[1] = __builtin_bit_cast(u16x8, lo);
  } else {
    f32x16 rest;
#pragma unroll
    for (int e = 0; e < 8; e++) rest[e] = s[base + e];
#pragma unroll
    for (int p = 1; p < Split<T>::PARTS; p++) {
#pragma unroll
      for (int e = 0; e < 8; e++) rest[e] -= T::unpack(part[p - 1][e]);
      part[p] = pack8<T>(rest, 0);
    }
  }
}

template <typename T, int D, bool MASK>
__global__ __launch_bounds__(THREADS, 2) void sdpa_fwd_split(const u16* __restrict__ q, const u16* __restrict__ k,
                                                             const u16* __restrict__ v, const u16* __restrict__ mask,
                                                             u16* __restrict__ out, float* __restrict__ lse, int64_t batch, int t_q,
                                                             int t_k, int hd, int hd_v, float scale) {
  __shared__ __attribute__((aligned(16))) u16 Ks[2][TILE * tile_stride<D>()];
  __shared__ __attribute__((aligned(16))) u16 Vs[2][TILE * tile_stride<D>()];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, n = lane & 31;
  int64_t b, qb;
  head_and_block(batch, (t_q + 127) / 128, b, qb);
  const int row = (int)qb * 128 + wave * 32 + n;
  const Rows qrows(q + b * (int64_t)t_q * hd, t_q, hd);
  const Rows krows(k + b * (int64_t)t_k * hd, t_k, hd), vrows(v + b * (int64_t)t_k * hd_v, t_k, hd_v);
  const MaskRow mrow(MASK ? mask + b * (int64_t)t_k : nullptr, MASK ? t_k : 0);
  typedef Split<T> P;
  const float c2 = scale * LOG2E, lift = P::LAG / c2;

  u16x8 qf[D / 16];
  f32x16 acc[P::TOTALS][D / 32];
  float m = neg_inf(), l = 0.f;
#pragma unroll
  for (int ds = 0; ds < D / 16; ds++) qf[ds] = qrows.load8(ds * 16 + 8 * h < hd ? row * hd + ds * 16 + 8 * h : 0x3f000000);
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < P::TOTALS; t++)
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++) acc[t][dt] = zero16();
  };
  clear();

  const int ntiles = (t_k + TILE - 1) / TILE;
  __shared__ int broken;
  if (threadIdx.x == 0) broken = 0;  // the first barrier of walk orders it
  auto walk = [&](auto first) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(first)::value;
    WidthStage<D> st;
    st.template load<T, MASK>(krows, vrows, hd, hd_v, mrow, 0);
    st.store(Ks[0], Vs[0]);
    if (ntiles > 1) st.template load<T, MASK>(krows, vrows, hd, hd_v, mrow, TILE);
    u16 mnext = MASK ? mrow.load(lane) : (u16)0;
    __syncthreads();
    for (int it = 0; it < ntiles; it++) {
      const int k0 = it * TILE, buf = it & 1;
      const u16* Kt = Ks[buf];
      const u16* Vt = Vs[buf];
      uint64_t live = ~0ull;
      if (MASK) {
        live = live_keys<T>(mnext);
        if (it + 1 < ntiles) mnext = mrow.load(k0 + TILE + lane);
      }
      f32x16 s[2] = {zero16(), zero16()};
#pragma unroll
      for (int ds = 0; ds < D / 16; ds++)
#pragma unroll
        for (int sub = 0; sub < 2; sub++) s[sub] = T::mfma32(read_row<D>(Kt, sub * 32 + n, 2 * ds + h), qf[ds], s[sub]);
      if (k0 + TILE > t_k || (MASK && live != ~0ull)) {
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
          const unsigned mb = (unsigned)(live >> (sub * 32 + 4 * h));
#pragma unroll
          for (int i = 0; i < 16; i++) s[sub][i] = hidden<false, MASK>(k0, sub, i, h, t_k, row, mb) ? neg_inf() : s[sub][i];
        }
      }
      if constexpr (SPLIT) {
        float mx = neg_inf();
#pragma unroll
        for (int sub = 0; sub < 2; sub++)
#pragma unroll
          for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[sub][i]);
        mx = pair_max(mx);
        if (__any(mx - m > lift)) {  // the reference point moves as in sdpa_fwd_mfma
          const float mnew = fmaxf(m, mx);
          const float alpha = mnew == neg_inf() ? 1.f : fast_exp2((m - mnew) * c2);
          l *= alpha;
#pragma unroll
          for (int t = 0; t < P::TOTALS; t++)
#pragma unroll
            for (int dt = 0; dt < D / 32; dt++) acc[t][dt] *= alpha;
          m = mnew;
        }
      }
      const float at = m == neg_inf() ? 0.f : m;
      float base = at * c2 - P::SHIFT;
      if (__any(fabsf(at * c2) > FAR)) {  // the scores less the reference point first, rounded at their own size
#pragma unroll
        for (int sub = 0; sub < 2; sub++)
#pragma unroll
          for (int i = 0; i < 16; i++) s[sub][i] -= at;
        base = -P::SHIFT;
      }
      float rs = 0.f;
#pragma unroll
      for (int sub = 0; sub < 2; sub++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          s[sub][i] = fast_exp2(fmaf(s[sub][i], c2, -base));
          rs += s[sub][i];
          if constexpr (!SPLIT) s[sub][i] = s[sub][i] > 0.f ? 0x1p-14f : s[sub][i];
        }
      if constexpr (SPLIT) l += rs;
#pragma unroll
      for (int sub = 0; sub < 2; sub++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          u16x8 part[P::PARTS];
          split8<T>(s[sub], 8 * c, part);
#pragma unroll
          for (int dt = 0; dt < D / 32; dt++) {
            const u16x8 vt = read_transposed<D>(Vt, sub * 32 + 16 * c, dt * 32);
#pragma unroll
            for (int p = 0; p < (SPLIT ? P::PARTS : 1); p++) acc[p % P::TOTALS][dt] = T::mfma32(vt, part[p], acc[p % P::TOTALS][dt]);
          }
        }
      if (it + 1 < ntiles) {
        st.store(Ks[buf ^ 1], Vs[buf ^ 1]);
        if (it + 2 < ntiles) st.template load<T, MASK>(krows, vrows, hd, hd_v, mrow, k0 + 2 * TILE);
      }
      __syncthreads();
    }
  };
  walk(std::true_type{});
  const float total = pair_sum(l);
  const float mul = 1.f / total;
  if constexpr (P::TOTALS == 2) {
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[0][dt][i] = fmaf(acc[1][dt][i], 0x1p-12f, acc[0][dt][i]);
  }
  u16* o = out + (b * (int64_t)t_q + row) * hd_v;
  bool nan = false;
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) nan |= acc[0][dt][i] != acc[0][dt][i];
  if (nan && row < t_q) broken = 1;
  if (row < t_q) {
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int d = dt * 32 + 8 * g + 4 * h;
        if (d < hd_v) *(u16x4*)(o + d) = u16x4{T::pack(acc[0][dt][4 * g] * mul), T::pack(acc[0][dt][4 * g + 1] * mul), T::pack(acc[0][dt][4 * g + 2] * mul), T::pack(acc[0][dt][4 * g + 3] * mul)};
    }
    if (h == 0) lse[b * (int64_t)t_q + row] = m * scale + logf(total * __builtin_exp2f(-P::SHIFT));
  }
  __syncthreads();
  if (!broken) return;
  clear();
  walk(std::false_type{});
  if (row >= t_q) return;
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int d = dt * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      if (d < hd_v && !(fabsf(acc[0][dt][i]) < __builtin_inff())) o[d] = T::pack(acc[0][dt][i]);
    }
}

template <typename T, int D>
int launch_split(const SdpaArgs& a) {
  const int64_t blocks = a.batch * ((a.t_q + 127) / 128);
  if (blocks > 0x7fffffff) return fail(LIMN_HIP_EUNSUPPORTED, "sdpa: %lld workgroups exceed one launch", (long long)blocks);
  const dim3 grid((unsigned)blocks), block(THREADS);
  if (a.mask != nullptr)
    hipLaunchKernelGGL((sdpa_fwd_split<T, D, true>), grid, block, 0, a.stream, (const u16*)a.q, (const u16*)a.k, (const u16*)a.v,
                       (const u16*)a.mask, (u16*)a.out0, (float*)a.out1, a.batch, (int)a.t_q, (int)a.t_k, (int)a.hd, (int)a.hd_v, (float)a.scale);
  else
    hipLaunchKernelGGL((sdpa_fwd_split<T, D, false>), grid, block, 0, a.stream, (const u16*)a.q, (const u16*)a.k, (const u16*)a.v,
                       (const u16*)nullptr, (u16*)a.out0, (float*)a.out1, a.batch, (int)a.t_q, (int)a.t_k, (int)a.hd, (int)a.hd_v, (float)a.scale);
  return check_hip(hipGetLastError(), "launching an sdpa kernel");
}

template <typename T>
int launch_split_width(const SdpaArgs& a) {
  const int64_t width = a.hd > a.hd_v ? a.hd : a.hd_v;
  if (width <= 32) return launch_split<T, 32>(a);
  if (width <= 64) return launch_split<T, 64>(a);
  if (width <= 96) return launch_split<T, 96>(a);
  return launch_split<T, 128>(a);
}

}  // namespace

// Measured, us, float32 products (sdpa_wide.h) / these: f16, 256 heads, 197 x 1021, key mask, 80 dims
// 407/70, 32 dims 102/49, 16 dims 104/44; 12 heads 200 x 1000 x 80 58/32; 64 x 128 x 128 x 96 14/8. At up
// to 32 dims a few workgroups of 128 queries are no faster than waves that share out the keys: 1 head
// 64 x 4096 x 32 63/67, 4 heads 33 x 77 x 32 6.1/6.8.
bool split_takes(SdpaPass pass, const SdpaArgs& a) {
  if (pass != SDPA_FWD || a.causal) return false;
  if (!(a.scale >= 0x1p-64 && a.scale <= 0x1p64)) return false;  // scale log2(e) and its inverse, as floats, neither 0 nor infinite
  if (a.dtype != LIMN_HIP_FLOAT16 && a.dtype != LIMN_HIP_BFLOAT16) return false;
  if (a.hd % 8 != 0 || a.hd_v % 8 != 0 || a.hd > 128 || a.hd_v > 128) return false;
  const int64_t width = a.hd > a.hd_v ? a.hd : a.hd_v, rows = a.t_q > a.t_k ? a.t_q : a.t_k;
  if ((rows + 256) * width >= 0x3f000000) return false;  // element offsets below the one that reads zeros
  if (width <= 32 && a.batch * ((a.t_q + 127) / 128) < 16) return false;
  const uintptr_t in = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v;
  return in % 4 == 0 && (uintptr_t)a.out0 % 8 == 0;
}

int launch_sdpa_split(const SdpaArgs& a) {
  return a.dtype == LIMN_HIP_FLOAT16 ? launch_split_width<F16>(a) : launch_split_width<BF16>(a);
}

}  // namespace limn
