// Dense float32 contraction on CDNA4 matrix cores: C[b, m, n] = sum_k A[b, m, k] * B[b, k, n] with
// v_mfma_f32_32x32x2f32 (float32 operands and products, float32 totals) and an optional relu, bias
// and residual at the store. float32 is limn's default type, so this is what a Linear layer and its
// gradients become unless a model casts them down.
//
// What bounds it: the float32 matrix rate, 1/16 of the bf16 one (157 TFLOP/s; one 32x32x2 product
// holds a SIMD's matrix core for 64 cycles). LDS and memory have slack, so operands take the plain
// route, memory -> registers -> LDS, with any row stride and alignment: a float buffer load of 16
// bytes needs 4-byte alignment only, and the buffer's range check is per dword, so a chunk that
// straddles an operand's end reads its valid part and zeros.
//
// Tiles: 128 x 128 (4 waves of 64 x 64) or 64 x 64 (4 waves of 32 x 32), see plan_f32, with k split
// into slices while the tiles are too few; the slices' partial tiles go to a workspace and are added
// per element in slice order, so results do not depend on scheduling. k advances 32 per stage through two LDS buffers, one
// barrier per stage, the next stage's loads in flight under the current one's products.
//
// LDS tiles keep their memory orientation. k-contiguous: [rows][32 + 4], a lane takes the four k
// values 8g + 4 (lane / 32) + j, j = 0..3, of its row with one ds_read_b128 and step j multiplies
// the j-th of them (k may be summed in any order as long as both operands agree).
// Row-contiguous: [32][rows + 8], the same k values by four ds_read_b32, the two 32-lane halves
// four LDS rows and so half the banks apart.
//
// Accuracy: the product adds its terms one after another, each sum rounded, so a running total's error
// grows with the square root of its length; every two stages (64 k) the accumulators are added to a
// second set and start again from zero. Where the general reduce kernels hold many partial sums (an
// operand contiguous along k, or few cells) the 64 also go in four chains of 16, at some 5% of the time;
// where those kernels add all of k in one thread (a weight gradient) in one. Off float64, relative to the
// result, general kernels / these: x @ w^T at k = 512 1.0e-7/1.0e-7, 2048 1.3e-7/1.1e-7; x^T @ y over 256
// rows 2.9e-7/1.5e-7, over 2048 8.1e-7/1.6e-7.
//
// Measured figures are at plan_f32 below and at F32_PAYS (matmul.h).

#include <type_traits>

#include "matmul.h"

namespace limn {

// Four chains a cell where the general kernels sum as closely (see the accuracy note).
static bool f32_chains(const MatmulShape& s) {
  return s.a_k == 1 || s.b_k == 1 || s.batch * s.M * s.N < ((int64_t)1 << 18);
}

namespace {

constexpr int FB = 32;    // k per stage
constexpr int FTHREADS = 256;

template <int ROWS, bool KCONTIG>
struct F32Operand {
  static constexpr int STRIDE = KCONTIG ? FB + 4 : ROWS + 8;
  static constexpr int ELEMS = STRIDE * (KCONTIG ? ROWS : FB);
  static constexpr int PER_ROW = KCONTIG ? FB / 4 : ROWS / 4;   // 16-byte chunks per LDS row
  static constexpr int LOADS = ROWS * FB / 4 / FTHREADS;
  __amdgpu_buffer_rsrc_t rsrc;
  int stride, row0;
  f32x4 r[LOADS];

  // the resource spans the operand's batch slice exactly: rows and k past its end read as zeros
  __device__ __forceinline__ F32Operand(const float* base, int64_t rows, int64_t depth, int64_t stride_, int64_t row0_) {
    stride = (int)stride_;
    row0 = (int)row0_;
    const int64_t extent = KCONTIG ? (rows - 1) * stride_ + depth : (depth - 1) * stride_ + rows;
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)(extent * 4), 0x00020000);
  }

  __device__ __forceinline__ void load(int k0, int depth) {
#pragma unroll
    for (int s = 0; s < LOADS; s++) {
      const int c = threadIdx.x + s * FTHREADS;
      const int lrow = c / PER_ROW, lcol = (c % PER_ROW) * 4;
      const int off = KCONTIG ? (row0 + lrow) * stride + k0 + lcol : (k0 + lrow) * stride + row0 + lcol;
      r[s] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off * 4, 0, 0));
    }
  }

  // zero what a stage past `depth` read: a k-contiguous row runs on into the next row there, and
  // overlapping rows (a sliding window's strides) into other k
  __device__ __forceinline__ void clear_tail(int k0, int depth) {
#pragma unroll
    for (int s = 0; s < LOADS; s++) {
      const int c = threadIdx.x + s * FTHREADS;
      const int lrow = c / PER_ROW, lcol = (c % PER_ROW) * 4;
#pragma unroll
      for (int e = 0; e < 4; e++)
        if ((KCONTIG ? k0 + lcol + e : k0 + lrow) >= depth) r[s][e] = 0.f;
    }
  }

  __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
    for (int s = 0; s < LOADS; s++) {
      const int c = threadIdx.x + s * FTHREADS;
      *(f32x4*)(lds + (c / PER_ROW) * STRIDE + (c % PER_ROW) * 4) = r[s];
    }
  }

  // lane l gets X[row + l % 32][8g + 4 (l / 32) + j], j = 0..3
  __device__ __forceinline__ f32x4 operand(const float* lds, int row, int g) const {
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    if (KCONTIG) return *(const f32x4*)(lds + (row + n) * STRIDE + 8 * g + 4 * h);
    const float* p = lds + (8 * g + 4 * h) * STRIDE + row + n;
    return f32x4{p[0], p[STRIDE], p[2 * STRIDE], p[3 * STRIDE]};
  }
};

// out = res + (relu?(sum) + bias[n]), each addition rounded on its own
__device__ __forceinline__ float f32_terms(float v, int relu, const MatmulAddends& add, int64_t bz, int64_t row, int64_t col) {
  if (relu) v = v > 0.f ? v : 0.f;
  if (add.bias != nullptr) v = v + ((const float*)add.bias)[col * add.bias_n];
  if (add.res != nullptr) v = ((const float*)add.res)[bz * add.r_batch + row * add.r_m + col * add.r_n] + v;
  return v;
}

template <int BT, int CH, bool A_K, bool B_K, bool PARTIAL>
__global__ __launch_bounds__(FTHREADS, BT == 128 ? 2 : CH == 4 ? 3 : 4) void matmul_f32(const float* __restrict__ a, const float* __restrict__ b,
                                                                          float* __restrict__ c, MatmulShape s, int64_t chunk,
                                                                          int wide, int relu, MatmulAddends add) {
  constexpr int T = BT / 64;  // 32 x 32 accumulators per wave along m and along n
  using OA = F32Operand<BT, A_K>;
  using OB = F32Operand<BT, B_K>;
  __shared__ __attribute__((aligned(16))) float As[2][OA::ELEMS];
  __shared__ __attribute__((aligned(16))) float Bs[2][OB::ELEMS];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, n32 = lane & 31;
  const int wm = (wave >> 1) * (BT / 2), wn = (wave & 1) * (BT / 2);
  const int64_t tiles_n = (s.N + BT - 1) / BT, tiles_m = (s.M + BT - 1) / BT;
  const int64_t per_batch = tiles_m * tiles_n, per_slice = s.batch * per_batch;
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles, walked in groups of
  // 4 tile rows so that its L2 holds few operand rows and columns
  int64_t id = blockIdx.x;
  if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
  const int64_t slice = id / per_slice;
  const int64_t bz = (id - slice * per_slice) / per_batch;
  const int64_t t = id - slice * per_slice - bz * per_batch;
  constexpr int64_t GROUP = 4;
  const int64_t group = t / (GROUP * tiles_n), first = group * GROUP;
  const int64_t rows = tiles_m - first < GROUP ? tiles_m - first : GROUP;
  const int64_t tm = first + (t - group * GROUP * tiles_n) % rows, tn = (t - group * GROUP * tiles_n) / rows;
  const int64_t m0 = tm * BT, n0 = tn * BT;
  const int k_lo = (int)(slice * chunk), depth = (int)(slice * chunk + chunk < s.K ? slice * chunk + chunk : s.K);

  f32x16 acc[CH][T][T], total[T][T];
#pragma unroll
  for (int i = 0; i < T; i++)
#pragma unroll
    for (int j = 0; j < T; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) total[i][j][e] = 0.f;

  OA oa(a + bz * s.a_batch, s.M, s.K, A_K ? s.a_m : s.a_k, m0);
  OB ob(b + bz * s.b_batch, s.N, s.K, B_K ? s.b_n : s.b_k, n0);
  const int stages = (depth - k_lo + FB - 1) / FB;
  oa.load(k_lo, depth);
  ob.load(k_lo, depth);
  if (k_lo + FB > depth) {
    oa.clear_tail(k_lo, depth);
    ob.clear_tail(k_lo, depth);
  }
  oa.store(As[0]);
  ob.store(Bs[0]);
  __syncthreads();
  // one stage from LDS buffer `cur` while the next is loaded, then stored to the other; `fresh` starts
  // the accumulators from zero (as the product's constant third operand)
  auto stage = [&](auto fresh, int st, int cur) __attribute__((always_inline)) {
    const float* at = As[cur];
    const float* bt = Bs[cur];
    const int next = k_lo + (st + 1) * FB;
    if (st + 1 < stages) {
      oa.load(next, depth);
      ob.load(next, depth);
    }
#pragma unroll
    for (int g = 0; g < FB / 8; g++) {
      f32x4 av[T], bv[T];
#pragma unroll
      for (int i = 0; i < T; i++) av[i] = oa.operand(at, wm + i * 32, g);
#pragma unroll
      for (int j = 0; j < T; j++) bv[j] = ob.operand(bt, wn + j * 32, g);
      // the B operand goes first: an accumulator then holds C transposed, 4 consecutive n per lane
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
          for (int j = 0; j < T; j++) {
            f32x16& c = acc[q % CH][i][j];
            f32x16 from = c;
            if (decltype(fresh)::value && g == 0 && q < CH) {
#pragma unroll
              for (int e = 0; e < 16; e++) from[e] = 0.f;
            }
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[j][q], av[i][q], from, 0, 0, 0);
          }
    }
    if (st + 1 < stages) {
      if (next + FB > depth) {
        oa.clear_tail(next, depth);
        ob.clear_tail(next, depth);
      }
      oa.store(As[cur ^ 1]);
      ob.store(Bs[cur ^ 1]);
    }
    __syncthreads();
  };
  for (int st = 0; st < stages; st += 2) {
    stage(std::true_type{}, st, 0);
    if (st + 1 < stages) stage(std::false_type{}, st + 1, 1);
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          total[i][j][e] += CH == 4 ? (acc[0][i][j][e] + acc[1 % CH][i][j][e]) + (acc[2 % CH][i][j][e] + acc[3 % CH][i][j][e]) : acc[0][i][j][e];
  }

  // lane holds C[m = wm + 32 i + n32][n = wn + 32 j + 8 q + 4 h + e], e = 0..3
#pragma unroll
  for (int i = 0; i < T; i++) {
    const int64_t row = m0 + wm + i * 32 + n32;
    if (row >= s.M) continue;
#pragma unroll
    for (int j = 0; j < T; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int64_t col = n0 + wn + j * 32 + 8 * q + 4 * h;
        if (col >= s.N) continue;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = total[i][j][4 * q + e];
        float* o = PARTIAL ? c + ((slice * s.batch + bz) * s.M + row) * s.N + col : c + bz * s.c_batch + row * s.c_m + col * s.c_n;
        if (!PARTIAL) {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (col + e < s.N) v[e] = f32_terms(v[e], relu, add, bz, row, col + e);
        }
        if (wide && col + 3 < s.N) {
          *(f32x4*)o = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (col + e < s.N) o[e * (PARTIAL ? 1 : s.c_n)] = v[e];
        }
      }
  }
}

// The slices of a split contraction added per element in slice order, then the terms and the store.
__global__ __launch_bounds__(256) void matmul_f32_splits(const float* __restrict__ ws, float* __restrict__ c, MatmulShape s,
                                                         int64_t split, int relu, MatmulAddends add) {
  const int64_t total = s.batch * s.M * s.N;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    float v = ws[i];
    for (int64_t k = 1; k < split; k++) v += ws[k * total + i];
    const int64_t col = i % s.N, row = (i / s.N) % s.M, bz = i / (s.N * s.M);
    c[bz * s.c_batch + row * s.c_m + col * s.c_n] = f32_terms(v, relu, add, bz, row, col);
  }
}

#define LIMN_F32_INSTANCE(BT, CH, AK, BKC, P)                                                                             \
  template __global__ void matmul_f32<BT, CH, AK, BKC, P>(const float* __restrict__, const float* __restrict__, float* __restrict__, \
                                                          MatmulShape, int64_t, int, int, MatmulAddends);
#define LIMN_F32_LAYOUT(BT, CH, P) \
  LIMN_F32_INSTANCE(BT, CH, true, true, P) LIMN_F32_INSTANCE(BT, CH, true, false, P) LIMN_F32_INSTANCE(BT, CH, false, true, P) LIMN_F32_INSTANCE(BT, CH, false, false, P)
LIMN_F32_LAYOUT(128, 1, false)
LIMN_F32_LAYOUT(64, 1, false)
LIMN_F32_LAYOUT(64, 1, true)
LIMN_F32_LAYOUT(64, 4, false)
LIMN_F32_LAYOUT(64, 4, true)
#undef LIMN_F32_LAYOUT
#undef LIMN_F32_INSTANCE

template <int BT, int CH, bool A_K, bool B_K, bool PARTIAL>
int launch_tiles(const float* a, const float* b, float* c, const MatmulShape& s, const MatmulPlan& plan, int relu,
                 const MatmulAddends& add, hipStream_t stream) {
  const int64_t blocks = plan.split * s.batch * ((s.M + BT - 1) / BT) * ((s.N + BT - 1) / BT);
  if (blocks > 0x7fffffff) return fail(LIMN_HIP_EUNSUPPORTED, "contract: %lld workgroups exceed one launch", (long long)blocks);
  const bool rows16 = s.c_n == 1 && s.c_m % 4 == 0 && s.c_batch % 4 == 0;
  const int wide = (uintptr_t)c % 16 == 0 && (PARTIAL ? s.N % 4 == 0 : rows16);
  hipLaunchKernelGGL((matmul_f32<BT, CH, A_K, B_K, PARTIAL>), dim3((unsigned)blocks), dim3(FTHREADS), 0, stream, a, b, c, s,
                     plan.chunk, wide, relu, add);
  return check_hip(hipGetLastError(), "launching the float32 contraction");
}

template <bool A_K, bool B_K>
int launch_layout(const float* a, const float* b, float* c, const MatmulShape& s, const MatmulPlan& plan, int relu,
                  const MatmulAddends& add, float* ws, hipStream_t stream) {
  if (plan.tile == 128) return launch_tiles<128, 1, A_K, B_K, false>(a, b, c, s, plan, relu, add, stream);
  const bool chains = f32_chains(s);
  if (plan.split == 1)
    return chains ? launch_tiles<64, 4, A_K, B_K, false>(a, b, c, s, plan, relu, add, stream)
                  : launch_tiles<64, 1, A_K, B_K, false>(a, b, c, s, plan, relu, add, stream);
  const int rc = chains ? launch_tiles<64, 4, A_K, B_K, true>(a, b, ws, s, plan, relu, add, stream)
                        : launch_tiles<64, 1, A_K, B_K, true>(a, b, ws, s, plan, relu, add, stream);
  if (rc != LIMN_HIP_OK) return rc;
  const int64_t total = s.batch * s.M * s.N;
  const int64_t blocks = (total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096;
  hipLaunchKernelGGL(matmul_f32_splits, dim3((unsigned)blocks), dim3(256), 0, stream, (const float*)ws, c, s, plan.split, relu, add);
  return check_hip(hipGetLastError(), "launching the float32 slice fold");
}

}  // namespace

bool f32_layout_ok(const MatmulShape& s) {
  // one stride of each operand 1, none negative; the kernel addresses a batch slice by 32-bit byte
  // offsets, and a tile or stage overhanging its end must still be addressable
  if (!(s.a_k == 1 || s.a_m == 1) || !(s.b_k == 1 || s.b_n == 1)) return false;
  if (s.a_m < 0 || s.a_k < 0 || s.b_n < 0 || s.b_k < 0 || s.a_batch < 0 || s.b_batch < 0) return false;
  auto reach = [](int64_t rows, int64_t depth, int64_t row_stride, int64_t k_stride) {
    return rows < ((int64_t)1 << 30) && depth < ((int64_t)1 << 30) && row_stride < ((int64_t)1 << 30) && k_stride < ((int64_t)1 << 30) &&
           ((double)(rows + 128) * row_stride + (double)(depth + 2 * FB) * k_stride + 256) * 4 < (double)INT32_MAX;
  };
  return reach(s.M, s.K, s.a_m, s.a_k) && reach(s.N, s.K, s.b_n, s.b_k);
}

// One chain: 128 x 128 tiles when there are two for every CU. Else 64 x 64, four to a CU. Those too few
// to give every CU two cut k: into slices of at least 512 up to four workgroups a CU, or, where slices
// that long cannot give every CU two, into slices of at least 128 that do. Measured, us (TFLOP/s), the
// general kernels before: (4096 x 512 -> 2048) 92 (93), 7000 before; (4096 x 2048 -> 512) 93 (92), its
// weight gradient over 4096 rows, four slices, 84 (102), 91 with two; 1024^3 two slices 31 (68), four
// 37; 2048^3 152 (113), 4096^3 x^T @ y 1080 (127; the matrix cores reach 154 in a large library product).
MatmulPlan plan_f32(const MatmulShape& s) {
  const int64_t t128 = s.batch * ((s.M + 127) / 128) * ((s.N + 127) / 128);
  const int64_t t64 = s.batch * ((s.M + 63) / 64) * ((s.N + 63) / 64);
  if (t128 >= 512 && !f32_chains(s)) return {128, 1, s.K};
  if (t64 >= 512) return {64, 1, s.K};
  int64_t split = 1024 / t64 < s.K / 512 ? 1024 / t64 : s.K / 512;
  if (split * t64 < 512) split = 512 / t64 < s.K / 128 ? 512 / t64 : s.K / 128;
  if (split <= 1) return {64, 1, s.K};
  int64_t chunk = (s.K + split - 1) / split;
  chunk = (chunk + FB - 1) / FB * FB;
  return {64, (s.K + chunk - 1) / chunk, chunk};
}

int64_t f32_workspace_bytes(const MatmulShape& s) {
  const MatmulPlan plan = plan_f32(s);
  return plan.split > 1 ? plan.split * s.batch * s.M * s.N * (int64_t)sizeof(float) : 0;
}

static int launch_matmul_f32_as(const void* a, const void* b, void* c, const MatmulShape& s, const MatmulPlan& plan, int epilogue,
                         const MatmulAddends& add, void* workspace, hipStream_t stream) {
  const bool a_k = s.a_k == 1, b_k = s.b_k == 1;
  const int relu = epilogue == MATMUL_EPILOGUE_RELU;
  const float *x = (const float*)a, *y = (const float*)b;
  float *o = (float*)c, *ws = (float*)workspace;
  if (a_k && b_k) return launch_layout<true, true>(x, y, o, s, plan, relu, add, ws, stream);
  if (a_k) return launch_layout<true, false>(x, y, o, s, plan, relu, add, ws, stream);
  if (b_k) return launch_layout<false, true>(x, y, o, s, plan, relu, add, ws, stream);
  return launch_layout<false, false>(x, y, o, s, plan, relu, add, ws, stream);
}

int launch_matmul_f32(const void* a, const void* b, void* c, MatmulShape s, int epilogue, const MatmulAddends& add,
                      void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  MatmulPlan plan = plan_f32(s);
  if (plan.split > 1 && (workspace == nullptr || workspace_bytes < f32_workspace_bytes(s))) plan = {64, 1, s.K};
  if (s.c_n != 1 && s.c_m == 1 && add.bias == nullptr) {
    // an output whose rows run along m: the product of the transposes, so that a lane's four
    // cells are neighbours in memory
    s = {s.batch, s.N, s.M, s.K, s.b_batch, s.b_n, s.b_k, s.a_batch, s.a_k, s.a_m, s.c_batch, s.c_n, s.c_m};
    MatmulAddends turned = add;
    turned.r_m = add.r_n;
    turned.r_n = add.r_m;
    const void* left = b;
    b = a;
    a = left;
    return launch_matmul_f32_as(a, b, c, s, plan, epilogue, turned, workspace, stream);
  }
  return launch_matmul_f32_as(a, b, c, s, plan, epilogue, add, workspace, stream);
}

}  // namespace limn
