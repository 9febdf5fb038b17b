// Host-side launchers of the prompt (prefill) kernels (qd_prefill.hip): the
// prompt's positions go through each layer together, as dense FP32 GEMMs on
// the matrix cores plus a causal GQA attention. The kernels take the one
// supported shape: hidden 896, 14 query heads over 2 KV heads of 64,
// intermediate 4864.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "qd_device.hpp"

namespace qd {

// Rows of FP32 values stored as their three BF16 parts (qd_gemm.hpp), one
// plane per part: a GEMM's left operand. `plane` is the stride between planes
// in elements (a multiple of 8).
struct PartRows {
  uint16_t *p;
  size_t plane;
  __host__ __device__ uint16_t *at(int row, int width) const { return p + static_cast<size_t>(row) * width; }
};

// Most k splits (partial products) of a GEMM.
constexpr int kGemmMaxSplits = 9;
// The k splits launch_gemm_partials should use for m rows (1 .. kGemmMaxSplits).
int gemm_splits(int m, int n, int k);

// partials[z][m][n] = slice z over k of A . W^T, for A [m][k] in parts and W
// [n][k] row-major in the storage type `dtype` (kWeights*). n a multiple of
// 128, k of 128.
hipError_t launch_gemm_partials(hipStream_t s, int dtype, const PartRows &a, int m, const float *w, int n, int k,
                                float *partials, int splits);

// act[r][i] = silu(A[r] . wg[i]) * (A[r] . wu[i]) for r < m, i < inter, in
// parts (inter a multiple of 64, k of 128).
hipError_t launch_gemm_swiglu(hipStream_t s, int dtype, const PartRows &a, int m, const float *wg, const float *wu,
                              int inter, int k, const PartRows &act);

// hidden[r] = embed[tokens[r]] and xn[r] = its RMSNorm with `gain`.
hipError_t launch_embed_norm(hipStream_t s, const float *embed, const uint32_t *tokens, int rows, const float *gain,
                             float eps, float *hidden, const PartRows &xn);

// hidden[r] += the sum of row r's partials, in slice order; with a gain also
// xn[r] = the RMSNorm of the new row.
hipError_t launch_residual_norm(hipStream_t s, const float *partials, int splits, int rows, float *hidden,
                                const float *gain, float eps, const PartRows &xn);

// Row r of q | k | v from its partials plus bias, rotated (rotate-half at
// position pos0 + r): q[r] and the cache rows pos0 + r.
hipError_t launch_qkv_rope(hipStream_t s, const float *partials, int splits, int rows, const float *bias, int pos0,
                           const float *rope_cos, const float *rope_sin, float *q, float *k_cache,
                           float *v_cache);

// Causal GQA attention of rows rotated queries at positions pos0.. over cache
// positions 0..pos0 + r (rows <= kAttnRecRows). records:
// kAttnRecRows * kAttnRecFloats floats of workspace for partial results.
constexpr int kAttnRecRows = 8192, kAttnRecFloats = 14 * (kHeadDim + 4);
hipError_t launch_attention_prefill(hipStream_t s, const float *q, int rows, int pos0, const float *k_cache,
                                    const float *v_cache, float *records, const PartRows &out);

}  // namespace qd
