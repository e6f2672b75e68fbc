// Internal launch interface of the dense-contraction kernel (matmul.hip).
#pragma once

#include "common.h"

namespace limn {

// C[b, m, n] = sum_k A[b, m, k] * B[b, k, n]; all strides in elements.
struct MatmulShape {
  int64_t batch, M, N, K;
  int64_t a_batch, a_m, a_k;
  int64_t b_batch, b_k, b_n;
  int64_t c_batch, c_m, c_n;
};

enum { MATMUL_EPILOGUE_NONE = 0, MATMUL_EPILOGUE_RELU = 1 };

// Terms added to the contraction after it is rounded to the output type, with one more rounding
// at the end: out = T(res[b, m, n] + (T(epilogue(sum)) + bias[n])), computed in float, either term
// left out when its pointer is null. This is an elementwise reader of the contraction that adds a
// bias vector (and a residual), evaluated at the store instead of in a launch of its own.
struct MatmulAddends {
  const void* bias;  // bias[n * bias_n], of the output type, or float32 rounded to it first
  int bias_f32;
  int64_t bias_n;
  const void* res;  // res[b * r_batch + m * r_m + n * r_n], of the output type
  int64_t r_batch, r_m, r_n;
  int vec;          // bit 0: bias_n == 1 and 16-byte aligned; bit 1: res rows the same (r_n == 1)
};

// How a contraction is cut: output tiles of `tile` x `tile`, k in `split` slices of `chunk`.
struct MatmulPlan {
  int tile;
  int64_t split, chunk;
};
MatmulPlan plan_matmul(const MatmulShape& s);
int64_t matmul_workspace_bytes(const MatmulShape& s);

// 1 when every operand is contiguous along one of its two dims with 16-byte aligned rows.
int matmul_layout_ok(const MatmulShape& s);
int launch_matmul(const void* a, const void* b, void* c, int dtype, const MatmulShape& s, int epilogue,
                  const MatmulAddends& add, void* workspace, int64_t workspace_bytes, hipStream_t stream);

// Products below which the general reduce kernels, whose one launch may also be merged with its
// neighbours, are never clearly the slower way. One call, us, general / contract (x @ w^T; x @ w; x^T @ y):
// float32 from 2^23 on by layout and shape (emit.contract_pays): (64 x 784 -> 128) 4.3/9.8, 5.9/10.2, 5.8/10.7;
// (32 x 512 -> 512) 16.4/8.4, 6.1/8.8, 5.6/9.2; (256 x 256 -> 256) 30.3/8.3, 43.7/8.6, 7.7/9.0; 512^3 226/11,
// 334/11, 40/12; 1024^3 1771/31, 3113/31, 260/31. Half widths pay for the copies: 257^3 14/15, 22/15, 9/15; 321^3 22/14, 75/14,
// 14/15; (65 x 8193 -> 65) 16/22, 130/21, 17/21; (129 x 4097 -> 129) 28/21, 251/21, 26/21; 513^3 68/18,
// 297/19, 46/19; 1025^3 651/29, 2697/30, 280/29. With a side under 64 the copy, padded to whole stages of
// 64, and the idle part of a tile can outweigh the product: (2^18 x 33 -> 33) 159/59, 123/59, 131/58, but
// (2^19 x 9 -> 9) 24/100, 28/99, 16/93 and (33 x 2^18 -> 33) 60/77, 862/103, 132/106.
constexpr double F32_PAYS = 1 << 23, PACK_PAYS = 1 << 26;
constexpr int64_t PACK_SIDE = 64;

// float32 operands and result (matmul_f32.hip), any row stride and alignment.
bool f32_layout_ok(const MatmulShape& s);
MatmulPlan plan_f32(const MatmulShape& s);
int64_t f32_workspace_bytes(const MatmulShape& s);
int launch_matmul_f32(const void* a, const void* b, void* c, MatmulShape s, int epilogue, const MatmulAddends& add,
                      void* workspace, int64_t workspace_bytes, hipStream_t stream);

// Half widths with any row alignment and any k, through aligned copies of the operands that need them
// (matmul_pack.hip). `shifted`: the operand does not start on a 16-byte boundary.
bool pack_layout_ok(const MatmulShape& s, bool a_shifted, bool b_shifted);
int64_t pack_workspace_bytes(const MatmulShape& s, bool a_shifted, bool b_shifted);
int launch_matmul_packed(const void* a, const void* b, void* c, int dtype, const MatmulShape& s, int epilogue,
                         const MatmulAddends& add, void* workspace, hipStream_t stream);

}  // namespace limn
