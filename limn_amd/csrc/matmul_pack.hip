// Half-width contractions whose operand rows are not 16-byte aligned, or whose k is no multiple of 8 (an
// odd width, ten classes, a shifted view): the operands that need it are first copied to aligned,
// zero-padded rows in the caller's workspace, then limn_hip_matmul's kernels run on the copies. They
// load 16 bytes at a time and need that; the copy reads and writes each such operand once, little beside
// the product, where the general reduce kernels take two 2-byte loads a product. bf16, us, general / this:
// (1235 x 1001) @ (1001 x 1235) 3847 / 31, (4099 x 2047) @ (2047 x 4099) 127310 / 136; more at PACK_PAYS
// (matmul.h).

#include "matmul.h"

namespace limn {
namespace {

struct Packed {
  bool need;
  int64_t batch, src_batch, src_row;
  unsigned rows, cols;          // the operand as rows of its contiguous dim
  unsigned dst_rows, dst_cols;  // its copy, dense
  unsigned blocks;              // of one batch entry's copy, 256 threads x 8 columns each; 0 when there is none
  const u16* src;
  u16* dst;
  int64_t bytes() const { return need ? (batch * dst_rows * dst_cols * 2 + 255) / 256 * 256 : 0; }
};

// dst[b][r][c] = src[b][r][c] inside (rows, cols), zero in the padding: both operands in one launch, a's
// blocks first, 8 columns (one 16-byte store) a thread. Bound by HBM: both
// operands of 4099 x 2047 and its transpose, 67 MB read and written, in 20 us (3.4 TB/s).
__global__ __launch_bounds__(256) void pack_rows(Packed a, Packed b) {
  const bool first = blockIdx.x < a.blocks;
  const Packed& p = first ? a : b;
  const unsigned i = (blockIdx.x - (first ? 0 : a.blocks)) * 256 + threadIdx.x, chunks = p.dst_cols / 8;
  const unsigned r = i / chunks, c = (i - r * chunks) * 8;
  if (r >= p.dst_rows) return;
  for (int64_t z = blockIdx.y; z < p.batch; z += gridDim.y) {
    u16x8 v;
#pragma unroll
    for (unsigned e = 0; e < 8; e++) v[e] = r < p.rows && c + e < p.cols ? p.src[z * p.src_batch + r * p.src_row + c + e] : (u16)0;
    *(u16x8*)(p.dst + (z * p.dst_rows + r) * p.dst_cols + c) = v;
  }
}

struct PackPlan {
  Packed a, b;
  MatmulShape s;  // the contraction of the copies
};

int64_t up(int64_t x, int64_t to) { return (x + to - 1) / to * to; }

// one operand: `other` is m or n, contiguous along k when kcontig
Packed pack_of(bool kcontig, int64_t batch, int64_t batch_stride, int64_t stride, int64_t other, int64_t K, int64_t Kp, bool shifted) {
  const int64_t extent = kcontig ? K : other;
  Packed p = {};
  p.need = shifted || K != Kp || stride % 8 != 0 || extent % 8 != 0 || batch_stride % 8 != 0;
  p.batch = batch_stride == 0 ? 1 : batch;
  p.src_batch = batch_stride;
  p.src_row = stride;
  p.rows = (unsigned)(kcontig ? other : K);
  p.cols = (unsigned)extent;
  p.dst_rows = (unsigned)(kcontig ? other : Kp);
  p.dst_cols = (unsigned)up(kcontig ? Kp : other, 8);
  p.blocks = p.need ? (unsigned)(((int64_t)p.dst_rows * (p.dst_cols / 8) + 255) / 256) : 0;
  return p;
}

PackPlan plan_pack(const MatmulShape& s, bool a_shifted, bool b_shifted) {
  const bool a_k = s.a_k == 1, b_k = s.b_k == 1;
  // A k of whole 8s stays as it is (the k-tail kernel takes it); else both copies pad it to whole stages.
  // A row-contiguous operand of a ragged width gets at least one padding row of k: the kernels' buffers
  // end with the last row's last element, inside a 16-byte load, and that row is then zeros either way.
  const bool ragged = (!a_k && s.M % 8 != 0) || (!b_k && s.N % 8 != 0);
  const int64_t Kp = s.K % 8 == 0 && !ragged ? s.K : up(s.K + ragged, 64);
  PackPlan p;
  p.a = pack_of(a_k, s.batch, s.a_batch, a_k ? s.a_m : s.a_k, s.M, s.K, Kp, a_shifted);
  p.b = pack_of(b_k, s.batch, s.b_batch, b_k ? s.b_n : s.b_k, s.N, s.K, Kp, b_shifted);
  p.s = s;
  p.s.K = Kp;
  if (p.a.need) {
    p.s.a_batch = s.a_batch == 0 ? 0 : p.a.dst_rows * p.a.dst_cols;
    (a_k ? p.s.a_m : p.s.a_k) = p.a.dst_cols;
  }
  if (p.b.need) {
    p.s.b_batch = s.b_batch == 0 ? 0 : p.b.dst_rows * p.b.dst_cols;
    (b_k ? p.s.b_n : p.s.b_k) = p.b.dst_cols;
  }
  return p;
}

// the copies' layout; a row-contiguous operand's padded rows count as rows of the contraction
MatmulShape padded(const PackPlan& p) {
  MatmulShape s = p.s;
  if (p.a.need && s.a_k != 1) s.M = p.a.dst_cols;
  if (p.b.need && s.b_k != 1) s.N = p.b.dst_cols;
  return s;
}

}  // namespace

bool pack_layout_ok(const MatmulShape& s, bool a_shifted, bool b_shifted) {
  if (!(s.a_k == 1 || s.a_m == 1) || !(s.b_k == 1 || s.b_n == 1)) return false;
  if (s.a_m < 1 || s.a_k < 1 || s.b_n < 1 || s.b_k < 1 || s.a_batch < 0 || s.b_batch < 0) return false;
  // the copies' rows and columns in 32 bits; the caller's strides need none
  if (s.M > INT32_MAX / 2 || s.N > INT32_MAX / 2 || s.K > INT32_MAX / 2) return false;
  return matmul_layout_ok(padded(plan_pack(s, a_shifted, b_shifted)));
}

int64_t pack_workspace_bytes(const MatmulShape& s, bool a_shifted, bool b_shifted) {
  const PackPlan p = plan_pack(s, a_shifted, b_shifted);
  return p.a.bytes() + p.b.bytes() + matmul_workspace_bytes(p.s);
}

int launch_matmul_packed(const void* a, const void* b, void* c, int dtype, const MatmulShape& s, int epilogue,
                         const MatmulAddends& add, void* workspace, hipStream_t stream) {
  PackPlan p = plan_pack(s, (uintptr_t)a % 16 != 0, (uintptr_t)b % 16 != 0);
  char* at = (char*)workspace;
  if (p.a.need) {
    p.a.src = (const u16*)a;
    p.a.dst = (u16*)at;
    a = at;
    at += p.a.bytes();
  }
  if (p.b.need) {
    p.b.src = (const u16*)b;
    p.b.dst = (u16*)at;
    b = at;
    at += p.b.bytes();
  }
  if (p.a.need || p.b.need) {
    const int64_t most = p.a.need && p.a.batch > p.b.batch || !p.b.need ? p.a.batch : p.b.batch;
    hipLaunchKernelGGL(pack_rows, dim3(p.a.blocks + p.b.blocks, (unsigned)(most < 65535 ? most : 65535)), dim3(256), 0, stream, p.a, p.b);
    const int rc = check_hip(hipGetLastError(), "launching the operand copies");
    if (rc != LIMN_HIP_OK) return rc;
  }
  return launch_matmul(a, b, c, dtype, p.s, epilogue, add, at, matmul_workspace_bytes(p.s), stream);
}

}  // namespace limn
