// Prompt (prefill) kernels for gfx950: the prompt's positions go through a
// layer together, so its projections are dense FP32 GEMMs on the BF16 matrix
// cores (operands split exactly into BF16 parts, qd_gemm.hpp) and its
// attention a causal flash attention (v_mfma_f32_16x16x4f32), instead of one
// decode step per position.
//
// Semantics follow the decode step per position (the reference's prompt
// stack, benchmarks/triton_mini_decoder_layer.cpp:811-849, is P sequential
// decode steps): RMSNorm eps, rotate-half RoPE at the absolute position,
// K/V cache rows written post-RoPE / raw, attention over positions
// 0..position inclusive with scale 1/sqrt(64) and query head h reading KV
// head h / (heads / kv_heads).
#include <hip/hip_runtime.h>

#include <cmath>
#include <algorithm>
#include <cstdint>

#include "qd_device.hpp"
#include "qd_device_math.hpp"
#include "qd_gemm.hpp"
#include "qd_prefill.hpp"

namespace qd {
namespace {

using namespace dev;

typedef float f4v __attribute__((ext_vector_type(4)));

// ---- row kernels: one prompt row per workgroup ---------------------------------

constexpr int kH = 896;      // hidden = query width
constexpr int kH4 = kH / 4;  // float4s of a row, one per thread of the first kH4

// The four values' parts to column 4 c of a row of planes.
__device__ __forceinline__ void put_parts(uint16_t *row, size_t plane, int c, float4 v) {
  const gemm::Parts a = gemm::split_value(v.x), b = gemm::split_value(v.y), d = gemm::split_value(v.z),
                    e = gemm::split_value(v.w);
#pragma unroll
  for (int p = 0; p < 3; ++p)
    *reinterpret_cast<uint2 *>(row + p * plane + 4 * c) =
        make_uint2(a.p[p] | uint32_t(b.p[p]) << 16, d.p[p] | uint32_t(e.p[p]) << 16);
}

// RMSNorm of a row held as one float4 per thread (threads c < kH4), x * inv *
// gain, as parts. (The decode kernels fold the norm past their GEMVs instead,
// inv * (W . (x * gain)); the two agree to rounding.)
__device__ __forceinline__ void norm_row(float4 v, const float *__restrict__ gain, float eps, uint16_t *row,
                                         size_t plane, float *red) {
  const int c = threadIdx.x;
  float s = c < kH4 ? fma4(v, v, 0.f) : 0.f;
  s = wave_sum(s);
  if (lane_id() == 0) red[wave_id()] = s;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < kWavesPerBlock; ++w) t += red[w];
  const float inv = rsqrtf(t / static_cast<float>(kH) + eps);
  if (c >= kH4) return;
  const float4 g = reinterpret_cast<const float4 *>(gain)[c];
  put_parts(row, plane, c, make_float4(v.x * inv * g.x, v.y * inv * g.y, v.z * inv * g.z, v.w * inv * g.w));
}

// Embedding row of each prompt token and its first norm.
__global__ __launch_bounds__(kBlock) void embed_norm_kernel(const float *__restrict__ embed,
                                                            const uint32_t *__restrict__ tokens,
                                                            const float *__restrict__ gain, float eps,
                                                            float *__restrict__ hidden, PartRows xn) {
  __shared__ float red[kWavesPerBlock];
  const int r = blockIdx.x, c = threadIdx.x;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c < kH4) {
    v = reinterpret_cast<const float4 *>(embed + static_cast<size_t>(tokens[r]) * kH)[c];
    reinterpret_cast<float4 *>(hidden + static_cast<size_t>(r) * kH)[c] = v;
  }
  norm_row(v, gain, eps, xn.at(r, kH), xn.plane, red);
}

// Sum of the `parts` split-K partials of float4 c of row r, in slice order:
// four are requested before any is added.
__device__ __forceinline__ float4 sum_partials(const float *__restrict__ part, size_t stride, size_t at, int parts) {
  constexpr int kBatch = 4;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int z0 = 0; z0 < parts; z0 += kBatch) {
    float4 p[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      p[j] = *reinterpret_cast<const float4 *>(part + static_cast<size_t>(min(z0 + j, parts - 1)) * stride + at);
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (z0 + j < parts) {
        v.x += p[j].x;
        v.y += p[j].y;
        v.z += p[j].z;
        v.w += p[j].w;
      }
  }
  return v;
}

// hidden row += the O or down GEMM's partials; then, with a gain, the next
// norm of the row.
__global__ __launch_bounds__(kBlock) void residual_norm_kernel(const float *__restrict__ part, int splits, int m,
                                                               float *__restrict__ hidden,
                                                               const float *__restrict__ gain, float eps,
                                                               PartRows xn) {
  __shared__ float red[kWavesPerBlock];
  const int r = blockIdx.x, c = threadIdx.x;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c < kH4) {
    float4 *h = reinterpret_cast<float4 *>(hidden + static_cast<size_t>(r) * kH) + c;
    const float4 s = sum_partials(part, static_cast<size_t>(m) * kH, static_cast<size_t>(r) * kH + 4 * c, splits);
    v = *h;
    v = make_float4(v.x + s.x, v.y + s.y, v.z + s.z, v.w + s.w);
    *h = v;
  }
  if (gain) norm_row(v, gain, eps, xn.at(r, kH), xn.plane, red);
}

// Packed QKV row r from the GEMM's partials plus bias, RoPE at position
// pos0 + r: the rotated query heads to q, the K/V rows to the cache.
constexpr int kQkv = kH + 4 * kHeadDim;  // q | two key heads | two value heads
__global__ __launch_bounds__(kBlock) void qkv_rope_kernel(const float *__restrict__ part, int splits, int m,
                                                          const float *__restrict__ bias, int pos0,
                                                          const float *__restrict__ rope_cos,
                                                          const float *__restrict__ rope_sin,
                                                          float *__restrict__ q, float *__restrict__ k_cache,
                                                          float *__restrict__ v_cache) {
  __shared__ __attribute__((aligned(16))) float4 row[kQkv / 4];
  const int r = blockIdx.x;
  for (int c = threadIdx.x; c < kQkv / 4; c += kBlock) {
    const float4 s = sum_partials(part, static_cast<size_t>(m) * kQkv, static_cast<size_t>(r) * kQkv + 4 * c, splits);
    const float4 b = reinterpret_cast<const float4 *>(bias)[c];
    row[c] = make_float4(s.x + b.x, s.y + b.y, s.z + b.z, s.w + b.w);
  }
  __syncthreads();
  constexpr int kHead4 = kHeadDim / 4, kHalf4 = kHead4 / 2, kKv4 = 2 * kHead4;  // float4s
  constexpr int kRotations = (kH / kHeadDim + 2) * kHalf4;
  static_assert(kRotations + kKv4 <= kBlock, "one item per thread");
  const int u = threadIdx.x;
  const size_t p = static_cast<size_t>(pos0) + r;
  if (u < kRotations) {
    const int head = u / kHalf4, i = u % kHalf4;
    const float4 a = row[head * kHead4 + i], b = row[head * kHead4 + kHalf4 + i];
    const float4 c = reinterpret_cast<const float4 *>(rope_cos + p * kRotary)[i];
    const float4 s = reinterpret_cast<const float4 *>(rope_sin + p * kRotary)[i];
    float4 x, y;
    rope_rotate(a.x, b.x, c.x, s.x, x.x, y.x);
    rope_rotate(a.y, b.y, c.y, s.y, x.y, y.y);
    rope_rotate(a.z, b.z, c.z, s.z, x.z, y.z);
    rope_rotate(a.w, b.w, c.w, s.w, x.w, y.w);
    constexpr int kHeads = kH / kHeadDim;
    float4 *dst = head < kHeads ? reinterpret_cast<float4 *>(q) + static_cast<size_t>(r) * kH4 + head * kHead4
                                : reinterpret_cast<float4 *>(k_cache) + p * kKv4 + (head - kHeads) * kHead4;
    dst[i] = x;
    dst[kHalf4 + i] = y;
  } else if (u < kRotations + kKv4) {
    reinterpret_cast<float4 *>(v_cache)[p * kKv4 + u - kRotations] = row[kH4 + kKv4 + u - kRotations];
  }
}

// ---- causal GQA flash attention ---------------------------------------------------
// One query block = (query head h, 16 prompt rows); a workgroup's four waves take
// the key blocks (32 positions) round-robin, each keeping an online softmax
// and an output accumulator for the 16 queries, merged in LDS at the end.
// Per key block a wave computes S = Q . K^T (two 16 x 16 tiles over 64
// dims) and O += P . V (four 16 x 16 tiles over 32 keys) with
// v_mfma_f32_16x16x4f32, whose lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[(l / 16) * 4 + r][l % 16] in register r.
constexpr int kQBlock = 16;
constexpr int kKBlock = 32;
constexpr int kKRow = kHeadDim + 4;   // LDS K row stride (conflict-free B reads)
constexpr int kVRow = kHeadDim + 16;  // LDS V row stride
constexpr int kPRow = kKBlock + 4;    // LDS P row stride

struct PrefillAttnLds {
  float k[kWavesPerBlock][kKBlock][kKRow];
  float v[kWavesPerBlock][kKBlock][kVRow];
  float p[kWavesPerBlock][kQBlock][kPRow];
  float ml[kWavesPerBlock][kQBlock][2];
  float o[kWavesPerBlock][kQBlock][kHeadDim + 1];
};

// Query block qb of head h (the causal extent of a block grows with qb).
__device__ __forceinline__ void attention_prefill_block(
    PrefillAttnLds &sh, int qb, const float *__restrict__ q, int rows, int pos0, int nq, int nkv,
    const float *__restrict__ k_cache, const float *__restrict__ v_cache, PartRows out) {
  const int h = blockIdx.y;
  const int r0 = qb * kQBlock;
  const int g = h / (nq / nkv);
  const int qd = nq * kHeadDim, kvd = nkv * kHeadDim;
  const int w = wave_id();
  const int lane = lane_id();
  const int lr = lane & 15, lg = lane >> 4;
  // Scores in base-2 units, s log2(e) / sqrt(64), so each softmax
  // exponential is one v_exp_f32 (2^x): e^(s / 8 - m) = 2^(s log2(e) / 8 - m').
  const float scale = 0.18033688011112042f;  // log2(e) / sqrt(64)
  const int last_row = min(rows, r0 + kQBlock) - 1;
  const int keys = pos0 + last_row + 1;  // causal extent of the block
  const int kblocks = (keys + kKBlock - 1) / kKBlock;

  // Query operand: lane supplies Q[row lr][dim 16 lg + s] at k-step s < 16
  // (the K operand takes the same dims), so each lane's 16 dims are
  // contiguous: four float4 reads.
  float qa[kHeadDim / 4];
  {
    const int qrow = min(r0 + lr, rows - 1);
    const float4 *q4 = reinterpret_cast<const float4 *>(q + static_cast<size_t>(qrow) * qd + h * kHeadDim + 16 * lg);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 v = q4[j];
      qa[4 * j] = v.x;
      qa[4 * j + 1] = v.y;
      qa[4 * j + 2] = v.z;
      qa[4 * j + 3] = v.w;
    }
  }
  // Running state of the lane's four query rows lg * 4 + r.
  float m[4], l[4];
  f4v o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.f;
    o[r] = f4v{0.f, 0.f, 0.f, 0.f};
  }
  float (*ks)[kKRow] = sh.k[w];
  float (*vs)[kVRow] = sh.v[w];
  float (*ps)[kPRow] = sh.p[w];
  // The block's K and V rows in registers: lane covers rows lane / 16 +
  // 4 i, float4 column lane % 16 (zeros past the causal extent). The wave's
  // next block is loaded while the current one is computed.
  float4 kr[kKBlock / 4], vr[kKBlock / 4];
  auto load_block = [&](int kb) {
#pragma unroll
    for (int i = 0; i < kKBlock / 4; ++i) {
      const int j = kb * kKBlock + lg + 4 * i;
      kr[i] = vr[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (j < keys) {
        kr[i] = *reinterpret_cast<const float4 *>(k_cache + static_cast<size_t>(j) * kvd + g * kHeadDim + 4 * lr);
        vr[i] = *reinterpret_cast<const float4 *>(v_cache + static_cast<size_t>(j) * kvd + g * kHeadDim + 4 * lr);
      }
    }
  };
  if (w < kblocks) load_block(w);
  for (int kb = w; kb < kblocks; kb += kWavesPerBlock) {
    const int k0 = kb * kKBlock;
    // Stage the block's rows in the wave's LDS, then start the next block's
    // loads.
#pragma unroll
    for (int i = 0; i < kKBlock / 4; ++i) {
      const int row = lg + 4 * i;
      const float4 kv = kr[i], vv = vr[i];
      *reinterpret_cast<float4 *>(&ks[row][4 * lr]) = kv;
      *reinterpret_cast<float4 *>(&vs[row][4 * lr]) = vv;
    }
    if (kb + kWavesPerBlock < kblocks) load_block(kb + kWavesPerBlock);
    // S tiles: keys k0 + 16 tt + lr. Every B operand is read from LDS before
    // the first MFMA (one wait instead of one per step), and the two tiles'
    // chains run interleaved; each chain keeps its order over st.
    float kop[2][kHeadDim / 4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const float4 v = *reinterpret_cast<const float4 *>(&ks[16 * tt + lr][16 * lg + 4 * j]);
        kop[tt][4 * j] = v.x;
        kop[tt][4 * j + 1] = v.y;
        kop[tt][4 * j + 2] = v.z;
        kop[tt][4 * j + 3] = v.w;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    f4v s[2] = {f4v{0.f, 0.f, 0.f, 0.f}, f4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int st = 0; st < kHeadDim / 4; ++st) {
      s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[st], kop[0][st], s[0], 0, 0, 0);
      s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[st], kop[1][st], s[1], 0, 0, 0);
    }
    // Online softmax per query row (row = lg * 4 + r, spread over the 16
    // lanes of DPP row lg and the two tiles).
    float corr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int qpos = pos0 + min(r0 + lg * 4 + r, rows - 1);
      float sv[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int key = k0 + 16 * tt + lr;
        sv[tt] = key <= qpos ? s[tt][r] * scale : -INFINITY;
      }
      const float m_new = fmaxf(m[r], row16_max(fmaxf(sv[0], sv[1])));
      float p0 = 0.f, p1 = 0.f;
      corr[r] = 1.f;
      if (m_new != -INFINITY) {
        p0 = __builtin_amdgcn_exp2f(sv[0] - m_new);
        p1 = __builtin_amdgcn_exp2f(sv[1] - m_new);
        corr[r] = __builtin_amdgcn_exp2f(m[r] - m_new);
      }
      l[r] = fmaf(l[r], corr[r], row16_sum(p0 + p1));
      m[r] = m_new;
      ps[lg * 4 + r][lr] = p0;
      ps[lg * 4 + r][16 + lr] = p1;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[dt][r] *= corr[r];
    // O += P . V: A = P[row lr][key 4 st + lg], B = V[key 4 st + lg][dim 16 dt + lr],
    // the operands read from LDS first as for S (this key order keeps the V
    // reads of the four lane groups on different banks).
    float pa[kKBlock / 4], vb[kKBlock / 4][4];
#pragma unroll
    for (int st = 0; st < kKBlock / 4; ++st) {
      pa[st] = ps[lr][4 * st + lg];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) vb[st][dt] = vs[4 * st + lg][16 * dt + lr];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < kKBlock / 4; ++st)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[st], vb[st][dt], o[dt], 0, 0, 0);
  }
  // Merge the four waves' partials.
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int q = lg * 4 + r;
    if (lr == 0) {
      sh.ml[w][q][0] = m[r];
      sh.ml[w][q][1] = l[r];
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) sh.o[w][q][16 * dt + lr] = o[dt][r];
  }
  __syncthreads();
  {
    const int q = threadIdx.x >> 4;        // 16 queries
    const int d0 = (threadIdx.x & 15) * 4;  // 4 dims each
    const int row = r0 + q;
    if (row < rows) {
      float mx = -INFINITY;
#pragma unroll
      for (int v = 0; v < kWavesPerBlock; ++v) mx = fmaxf(mx, sh.ml[v][q][0]);
      float den = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < kWavesPerBlock; ++v) {
        const float mv = sh.ml[v][q][0];
        const float f = mv == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mv - mx);
        den = fmaf(f, sh.ml[v][q][1], den);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(f, sh.o[v][q][d0 + e], acc[e]);
      }
      put_parts(out.at(row, qd) + h * kHeadDim, out.plane, d0 / 4,
                make_float4(acc[0] / den, acc[1] / den, acc[2] / den, acc[3] / den));
    }
  }
}

// Workgroup (pair p, head h) takes query blocks p and nqb - 1 - p: the pair's
// key blocks add up to about the same count for every p, so the launch is
// one balanced round of workgroups instead of a long causal tail.
__global__ __launch_bounds__(kBlock) void attention_prefill_kernel(
    const float *__restrict__ q, int rows, int pos0, int nq, int nkv,
    const float *__restrict__ k_cache, const float *__restrict__ v_cache, PartRows out) {
  __shared__ __attribute__((aligned(16))) PrefillAttnLds sh;
  const int nqb = (rows + kQBlock - 1) / kQBlock;
  const int p = blockIdx.x;
  attention_prefill_block(sh, p, q, rows, pos0, nq, nkv, k_cache, v_cache, out);
  const int p2 = nqb - 1 - p;
  if (p2 <= p) return;
  __syncthreads();  // the first block's merge has read the LDS
  attention_prefill_block(sh, p2, q, rows, pos0, nq, nkv, k_cache, v_cache, out);
}

// ---- GEMM launches ------------------------------------------------------------------

// Tile shapes of the split GEMM, by the number of rows.
enum Shape : int { kRows32K4 = 0, kRows32, kRows64, kRows128 };
struct ShapeInfo {
  int rows, cols, wk;
};
constexpr ShapeInfo kShapes[] = {{32, 32, 4}, {32, 64, 2}, {64, 128, 1}, {128, 128, 1}};
// The gate/up GEMM's 64-row shape splits k over two waves, not n.
constexpr ShapeInfo kSwiGLUShapes[] = {{32, 32, 4}, {32, 64, 2}, {64, 64, 2}, {128, 128, 1}};

// Up to 32 rows the waves split k, so that 32 columns make a workgroup;
// beyond, larger tiles reuse each staged weight for more rows as soon as there
// are enough of them to fill 256 CUs. us at m = 16 / 37 / 128 / 512 / 2048
// (128-row tile: 2048 only), gate/up: 12.2 / 20.4 / 31.4 with 32 rows and four
// k waves, 15.6 / 17.2 / 29.4 with two, 18.1 / 18.7 / 26.9 / 70 with 64 rows,
// 77 (512) / 237 (2048) with 128 rows (64 rows: 267 at 2048).
Shape gemm_shape(int m, bool swiglu) {
  if (m <= 32) return kRows32K4;
  if (m <= (swiglu ? 64 : 128)) return kRows32;
  return m <= 1024 ? kRows64 : kRows128;
}

template <int RB, int WM, int WN, int WK, typename W, bool kSwiGLU>
void launch_shape(hipStream_t s, const gemm::Args<W> &g) {
  const int mtiles = (g.m + 32 * RB * WM - 1) / (32 * RB * WM);
  const int pairs = g.n / ((kSwiGLU ? 16 : 32) * WN) * g.splits;
  const int grid = (pairs + gemm::kDealXcds - 1) / gemm::kDealXcds * gemm::kDealXcds * mtiles;
  gemm::gemm_split_kernel<RB, 1, WM, WN, WK, 2, W, kSwiGLU><<<grid, gemm::kThreads, 0, s>>>(g, mtiles, pairs);
}

template <typename W>
hipError_t launch_gemm_as(hipStream_t s, gemm::Args<W> g, bool swiglu) {
  const Shape shape = gemm_shape(g.m, swiglu);
  const ShapeInfo &i = (swiglu ? kSwiGLUShapes : kShapes)[shape];
  // Whole tiles of columns and whole slices of k (rows are masked).
  if (g.m <= 0 || g.k % (gemm::kSliceK * i.wk) != 0 || g.n % (swiglu ? i.cols / 2 : i.cols) != 0 ||
      g.splits < 1 || g.splits > g.k / (gemm::kSliceK * i.wk) || g.lda % 8 != 0 || g.a_plane % 8 != 0)
    return hipErrorInvalidValue;
  if (swiglu) {
    switch (shape) {
      case kRows32K4: launch_shape<1, 1, 1, 4, W, true>(s, g); break;
      case kRows32: launch_shape<1, 1, 2, 2, W, true>(s, g); break;
      case kRows64: launch_shape<2, 1, 2, 2, W, true>(s, g); break;
      case kRows128: launch_shape<4, 1, 4, 1, W, true>(s, g); break;
    }
  } else {
    switch (shape) {
      case kRows32K4: launch_shape<1, 1, 1, 4, W, false>(s, g); break;
      case kRows32: launch_shape<1, 1, 2, 2, W, false>(s, g); break;
      case kRows64: launch_shape<2, 1, 4, 1, W, false>(s, g); break;
      case kRows128: launch_shape<4, 1, 4, 1, W, false>(s, g); break;
    }
  }
  return hipGetLastError();
}

template <typename W>
hipError_t launch_gemm(hipStream_t s, const PartRows &a, int m, const float *w, const float *w2, int n, int k,
                       float *partials, int splits, const PartRows *act) {
  gemm::Args<W> g{};
  g.a = a.p;
  g.a_plane = a.plane;
  g.lda = k;
  g.w = reinterpret_cast<const W *>(w);
  g.w2 = reinterpret_cast<const W *>(w2);
  g.k = k;
  g.m = m;
  g.n = n;
  g.c = partials;
  g.splits = splits;
  if (act) {
    g.y = act->p;
    g.y_plane = act->plane;
  }
  return launch_gemm_as<W>(s, g, act != nullptr);
}

hipError_t launch_gemm(hipStream_t s, int dtype, const PartRows &a, int m, const float *w, const float *w2, int n,
                       int k, float *partials, int splits, const PartRows *act) {
  switch (dtype) {
    case kWeightsF32: return launch_gemm<float>(s, a, m, w, w2, n, k, partials, splits, act);
    case kWeightsBf16: return launch_gemm<Bf16>(s, a, m, w, w2, n, k, partials, splits, act);
    case kWeightsF16: return launch_gemm<F16>(s, a, m, w, w2, n, k, partials, splits, act);
  }
  return hipErrorInvalidValue;
}

}  // namespace

int gemm_splits(int m, int n, int k) {
  const ShapeInfo &i = kShapes[gemm_shape(m, false)];
  const int tiles = (m + i.rows - 1) / i.rows * (n / i.cols);
  // Enough workgroups for the 256 CUs, more where k is long (at m = 512 and
  // k = 4864: 32.7 us with 8 or 9 slices, 35.8 with 4; at k = 896: 13.2 with 3,
  // 13.3 with 7), each with at least one slice, and at most kGemmMaxSplits
  // partials for the row kernel to sum.
  const int want = ((k > 2048 ? 400 : 200) + tiles - 1) / tiles;
  return std::max(1, std::min({want, kGemmMaxSplits, k / (gemm::kSliceK * i.wk)}));
}

hipError_t launch_gemm_partials(hipStream_t s, int dtype, const PartRows &a, int m, const float *w, int n, int k,
                                float *partials, int splits) {
  if (!partials) return hipErrorInvalidValue;
  return launch_gemm(s, dtype, a, m, w, nullptr, n, k, partials, splits, nullptr);
}

hipError_t launch_gemm_swiglu(hipStream_t s, int dtype, const PartRows &a, int m, const float *wg, const float *wu,
                              int inter, int k, const PartRows &act) {
  return launch_gemm(s, dtype, a, m, wg, wu, inter, k, nullptr, 1, &act);
}

hipError_t launch_embed_norm(hipStream_t s, const float *embed, const uint32_t *tokens, int rows, const float *gain,
                             float eps, float *hidden, const PartRows &xn) {
  embed_norm_kernel<<<rows, kBlock, 0, s>>>(embed, tokens, gain, eps, hidden, xn);
  return hipGetLastError();
}

hipError_t launch_residual_norm(hipStream_t s, const float *partials, int splits, int rows, float *hidden,
                                const float *gain, float eps, const PartRows &xn) {
  residual_norm_kernel<<<rows, kBlock, 0, s>>>(partials, splits, rows, hidden, gain, eps, xn);
  return hipGetLastError();
}

hipError_t launch_qkv_rope(hipStream_t s, const float *partials, int splits, int rows, const float *bias, int pos0,
                           const float *rope_cos, const float *rope_sin, float *q, float *k_cache,
                           float *v_cache) {
  qkv_rope_kernel<<<rows, kBlock, 0, s>>>(partials, splits, rows, bias, pos0, rope_cos, rope_sin, q, k_cache,
                                          v_cache);
  return hipGetLastError();
}

hipError_t launch_attention_prefill(hipStream_t s, const float *q, int rows, int pos0, int nq, int nkv,
                                    const float *k_cache, const float *v_cache, const PartRows &out) {
  const int nqb = (rows + kQBlock - 1) / kQBlock;
  const dim3 grid((nqb + 1) / 2, nq);
  attention_prefill_kernel<<<grid, kBlock, 0, s>>>(q, rows, pos0, nq, nkv, k_cache, v_cache, out);
  return hipGetLastError();
}

}  // namespace qd
