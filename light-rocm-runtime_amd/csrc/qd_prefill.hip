// Prompt (prefill) kernels for gfx950: the prompt's positions go through a
// layer together, so its projections are dense FP32 GEMMs on the BF16 matrix
// cores (operands split exactly into BF16 parts, qd_gemm.hpp) and its
// attention a causal flash attention on the same split
// (v_mfma_f32_16x16x32_bf16), instead of one decode step per position.
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

#include "qd_attention.hpp"
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
// A workgroup takes 16 prompt rows of one KV group: a wave per query head of
// the group, which share each block of 64 keys, split once into BF16 parts in
// LDS. Both products run on v_mfma_f32_16x16x32_bf16 with the six products of
// qd_gemm.hpp, the leading one in its own accumulator:
//   S^T[key][row] = K . Q^T      A = K (lane: key l % 16, 8 dims from 8 (l / 16)),
//                                B = Q (row l % 16, the same dims)
//   O^T[dim][row] += V^T . P^T   A = V^T (dim l % 16), B = P (row l % 16)
// D holds element (4 (l / 16) + r, l % 16) in register r of lane l, so a lane
// keeps one prompt row throughout: its running maximum and rescale factor are
// its own, only the block maximum crosses lanes, and the probabilities of two
// 16-key tiles (keys 4 (l / 16) + r of each) are the B operand of the second
// product as they stand; V^T is laid out in LDS in that key order.
// What bounds it is the work per CU, not memory: a chunk of 512 rows is 64
// (row block, KV group) pairs, so each pair's key blocks are dealt to
// workgroups of `per_split` blocks whose partials a second kernel merges.
// Scores are in base-2 units, the query scaled by log2(e) / 8 (one v_exp_f32
// per exponential).
constexpr int kQRows = 16, kKeyBlock = 64, kGroupHeads = 7;
constexpr int kAttnWaves = kGroupHeads, kAttnThreads = kAttnWaves * kWave;
constexpr int kRec = kHeadDim + 4;        // partial record: m, l, two pad words, acc[64]
constexpr int kKv = 2 * kHeadDim;         // floats of a cache row
constexpr int kRowBytes = 2 * kHeadDim;   // an LDS row: 64 BF16 parts
constexpr int kKvPlane = kKeyBlock * kRowBytes;
static_assert(kHeadDim == kKeyBlock, "K and V^T rows are both 64 parts");

// 16-byte slot s of LDS row `row` (a key's dims or a dim's keys), so that the
// rows of sixteen consecutive lanes at one slot fall on distinct banks.
__device__ __forceinline__ int kv_slot(int row, int s) { return row * kRowBytes + 16 * (s ^ ((row >> 1) & 7)); }

// Maximum / sum over the four lanes l % 16 + 16 i, in each of them.
__device__ __forceinline__ void half_swap(float v, float &a, float &b) {
  a = b = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float quads_max(float v) {
  float a, b;
  half_swap(row_pair_max(v), a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float quads_sum(float v) {
  float a, b;
  half_swap(row_pair_sum(v), a, b);
  return a + b;
}

__device__ __forceinline__ f4v mfma16(gemm::bf8v a, gemm::bf8v b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
struct AttnArgs {
  const float *q;  // [rows][896]
  const float *k_cache, *v_cache;
  int rows, pos0, per_split, splits;
  float *rec;  // [rows][14][splits][kRec], splits > 1
  PartRows out;
};

// One head's attention of one prompt row over keys [k0, k1) in FP32, lane =
// dim, a key at a time: for a wave whose split products were not finite (an
// operand was not, or rounds to infinity in BF16).
__device__ void attention_row_fp32(const AttnArgs &g, int row, int head, int kv, int k0, int k1, float &m, float &l,
                                   float &acc) {
  const int d = lane_id();
  const float q = g.q[static_cast<size_t>(row) * kH + head * kHeadDim + d];
  m = -INFINITY;
  l = acc = 0.f;
  for (int key = k0; key < k1; ++key) {
    const size_t at = static_cast<size_t>(key) * kKv + kv * kHeadDim + d;
    const float score = wave_sum(q * g.k_cache[at]) * kScoreScaleLog2;
    if (score != -INFINITY) attn_fold(score, 1.f, g.v_cache[at], m, l, acc);
  }
}

__global__ __launch_bounds__(kAttnThreads, 4) void attention_prefill_kernel(AttnArgs g) {
  __shared__ __attribute__((aligned(16))) unsigned char kp[3 * kKvPlane], vp[3 * kKvPlane];
  const int r0 = blockIdx.x * kQRows, kv = blockIdx.y, z = blockIdx.z;
  const int keys = g.pos0 + min(g.rows, r0 + kQRows);  // causal extent of the row block
  const int k_begin = z * g.per_split * kKeyBlock;
  const int k_end = min(keys, k_begin + g.per_split * kKeyBlock);
  if (k_begin >= k_end) return;
  const int lane = lane_id(), head = kv * kGroupHeads + wave_id();
  const int lr = lane & 15, lg = lane >> 4;
  const int row = min(r0 + lr, g.rows - 1), pos = g.pos0 + row;

  // The block's K and V^T items of this thread (a block's are loaded when the
  // one before is done: the other workgroup of the CU fills the wait): item i <
  // 1024 is float4 i % 16 of key i / 16; 1024 + i is keys 4 (i / 64) .. + 3
  // of dim i % 64. Keys past the causal extent are zeros.
  constexpr int kItems = 2 * kKeyBlock * kHeadDim / 4, kPer = (kItems + kAttnThreads - 1) / kAttnThreads;
  float4 item[kPer];
  auto load = [&](int k0) {
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
      const int i = threadIdx.x + n * kAttnThreads;
      item[n] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i < kItems / 2) {
        const int key = k0 + i / 16;
        if (key < keys)
          item[n] = reinterpret_cast<const float4 *>(g.k_cache + static_cast<size_t>(key) * kKv + kv * kHeadDim)[i % 16];
      } else if (i < kItems) {
        const int key = k0 + 4 * ((i - kItems / 2) / 64);
        const float *v = g.v_cache + static_cast<size_t>(key) * kKv + kv * kHeadDim + i % 64;
        if (key < keys) item[n].x = v[0];
        if (key + 1 < keys) item[n].y = v[kKv];
        if (key + 2 < keys) item[n].z = v[2 * kKv];
        if (key + 3 < keys) item[n].w = v[3 * kKv];
      }
    }
  };
  auto stage = [&] {
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
      const int i = threadIdx.x + n * kAttnThreads;
      if (i >= kItems) break;
      uint2 p[3];
      gemm::split_pair(item[n].x, item[n].y, p[0].x, p[1].x, p[2].x);
      gemm::split_pair(item[n].z, item[n].w, p[0].y, p[1].y, p[2].y);
      unsigned char *dst;
      if (i < kItems / 2) {
        const int key = i / 16, d4 = i % 16;
        dst = kp + kv_slot(key, d4 / 2) + 8 * (d4 & 1);
      } else {
        // Keys 32 t + 16 h + 4 c .. + 3 are half h of slot 4 t + c.
        const int dim = i % 64, k4 = (i - kItems / 2) / 64;
        dst = vp + kv_slot(dim, 4 * (k4 >> 3) + (k4 & 3)) + 8 * ((k4 >> 2) & 1);
      }
#pragma unroll
      for (int u = 0; u < 3; ++u) *reinterpret_cast<uint2 *>(dst + u * kKvPlane) = p[u];
    }
  };
  gemm::bf8v qp[2][3];  // the wave's query rows, dims 32 s + 8 (l / 16) .. + 7
  {
    const float4 *q = reinterpret_cast<const float4 *>(g.q + static_cast<size_t>(row) * kH + head * kHeadDim);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const float4 a = q[8 * s + 2 * lg], b = q[8 * s + 2 * lg + 1];
      const float x[8] = {a.x * kScoreScaleLog2, a.y * kScoreScaleLog2, a.z * kScoreScaleLog2, a.w * kScoreScaleLog2,
                          b.x * kScoreScaleLog2, b.y * kScoreScaleLog2, b.z * kScoreScaleLog2, b.w * kScoreScaleLog2};
      gemm::split_eight(x, qp[s]);
    }
  }
  float m = -INFINITY, l = 0.f;  // l: this lane's share of the row's sum
  f4v lead[4], tail[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) lead[d] = tail[d] = f4v{0.f, 0.f, 0.f, 0.f};

  for (int k0 = k_begin; k0 < k_end; k0 += kKeyBlock) {
    load(k0);
    stage();
    __syncthreads();
    float p[4][4];
    // A tile of 16 keys at a time: more operands in flight would cost the
    // registers that let two workgroups share a CU.
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f4v sl = {0.f, 0.f, 0.f, 0.f}, st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        gemm::bf8v kx[3];
#pragma unroll
        for (int u = 0; u < 3; ++u)
          kx[u] = *reinterpret_cast<const gemm::bf8v *>(kp + u * kKvPlane + kv_slot(16 * t + lr, 4 * s + lg));
        sl = mfma16(kx[0], qp[s][0], sl);
        st = mfma16(kx[0], qp[s][1], st);
        st = mfma16(kx[1], qp[s][0], st);
        st = mfma16(kx[1], qp[s][1], st);
        st = mfma16(kx[0], qp[s][2], st);
        st = mfma16(kx[2], qp[s][0], st);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) p[t][r] = sl[r] + st[r];
      __builtin_amdgcn_sched_barrier(0);
    }
    if (k0 + kKeyBlock > g.pos0 + r0 + 1) {  // the block reaches past some row's position
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * t + 4 * lg + r > pos) p[t][r] = -INFINITY;
    }
    float mx = p[0][0];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, p[t][r]);
    mx = fmaxf(m, quads_max(mx));
    const float ref = mx == -INFINITY ? 0.f : mx;  // no key of the row yet: every term is 2^-inf = 0
    const float corr = exp2_fast(m - ref);
    m = mx;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[t][r] = exp2_fast(p[t][r] - ref);
        sum += p[t][r];
      }
    l = fmaf(l, corr, sum);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      lead[d] *= corr;
      tail[d] *= corr;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      gemm::bf8v px[3];
      const float x[8] = {p[2 * t][0],     p[2 * t][1],     p[2 * t][2],     p[2 * t][3],
                          p[2 * t + 1][0], p[2 * t + 1][1], p[2 * t + 1][2], p[2 * t + 1][3]};
      gemm::split_eight(x, px);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        gemm::bf8v vx[3];
#pragma unroll
        for (int u = 0; u < 3; ++u)
          vx[u] = *reinterpret_cast<const gemm::bf8v *>(vp + u * kKvPlane + kv_slot(16 * d + lr, 4 * t + lg));
        lead[d] = mfma16(vx[0], px[0], lead[d]);
        tail[d] = mfma16(vx[0], px[1], tail[d]);
        tail[d] = mfma16(vx[1], px[0], tail[d]);
        tail[d] = mfma16(vx[1], px[1], tail[d]);
        tail[d] = mfma16(vx[0], px[2], tail[d]);
        tail[d] = mfma16(vx[2], px[0], tail[d]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();  // the next block overwrites K and V
  }
  l = quads_sum(l);
  float probe = l * 0.f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    lead[d] += tail[d];
#pragma unroll
    for (int r = 0; r < 4; ++r) probe = fmaf(lead[d][r], 0.f, probe);
  }
  auto record = [&](int of_row) {
    return g.rec + ((static_cast<size_t>(of_row) * 2 * kGroupHeads + head) * g.splits + z) * kRec;
  };
  if (__builtin_amdgcn_ballot_w64(!(probe == 0.f)) != 0) {
    for (int i = 0; i < kQRows && r0 + i < g.rows; ++i) {
      float fm, fl, fa;
      attention_row_fp32(g, r0 + i, head, kv, k_begin, min(k_end, g.pos0 + r0 + i + 1), fm, fl, fa);
      if (g.splits > 1) {
        float *rec = record(r0 + i);
        rec[4 + lane] = fa;
        if (lane < 2) rec[lane] = lane == 0 ? fm : fl;
      } else {
        const gemm::Parts out = gemm::split_value(fa / fl);
        uint16_t *dst = g.out.at(r0 + i, kH) + head * kHeadDim + lane;
#pragma unroll
        for (int u = 0; u < 3; ++u) dst[u * g.out.plane] = out.p[u];
      }
    }
    return;
  }
  if (r0 + lr >= g.rows) return;
  // Lane: dims 16 d + 4 (l / 16) .. + 3 of its row.
  if (g.splits > 1) {
    float *rec = record(row);
#pragma unroll
    for (int d = 0; d < 4; ++d)
      *reinterpret_cast<float4 *>(rec + 4 + 16 * d + 4 * lg) = make_float4(lead[d][0], lead[d][1], lead[d][2], lead[d][3]);
    if (lg == 0) *reinterpret_cast<float2 *>(rec) = make_float2(m, l);
  } else {
#pragma unroll
    for (int d = 0; d < 4; ++d)
      put_parts(g.out.at(row, kH) + head * kHeadDim, g.out.plane, 4 * d + lg,
                make_float4(lead[d][0] / l, lead[d][1] / l, lead[d][2] / l, lead[d][3] / l));
  }
}

// One prompt row: the partials of its heads over the row block's splits.
__global__ __launch_bounds__(kBlock) void attention_merge_kernel(AttnArgs g) {
  const int row = blockIdx.x;
  const int keys = g.pos0 + min(g.rows, (row / kQRows + 1) * kQRows);
  const int splits = (keys + g.per_split * kKeyBlock - 1) / (g.per_split * kKeyBlock);
  const int head = threadIdx.x / (kHeadDim / 4), c = threadIdx.x % (kHeadDim / 4);
  if (head >= 2 * kGroupHeads) return;
  const float *rec = g.rec + (static_cast<size_t>(row) * 2 * kGroupHeads + head) * g.splits * kRec;
  // Eight records requested before any is used (a read at a time took 1 us
  // per split).
  constexpr int kBatch = 8;
  float m = -INFINITY, den = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int z0 = 0; z0 < splits; z0 += kBatch) {
    float2 ml[kBatch];
    float4 a[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const float *r = rec + min(z0 + j, splits - 1) * kRec;
      ml[j] = *reinterpret_cast<const float2 *>(r);
      a[j] = *reinterpret_cast<const float4 *>(r + 4 + 4 * c);
    }
    float mx = m;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) mx = fmaxf(mx, ml[j].x);
    const float ref = mx == -INFINITY ? 0.f : mx;
    const float corr = exp2_fast(m - ref);
    m = mx;
    den *= corr;
    acc = make_float4(acc.x * corr, acc.y * corr, acc.z * corr, acc.w * corr);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (z0 + j >= splits || (ml[j].x == -INFINITY && ml[j].y == 0.f)) continue;  // no key of the row in the split
      const float w = exp2_fast(ml[j].x - ref);
      den = fmaf(w, ml[j].y, den);
      acc = make_float4(fmaf(w, a[j].x, acc.x), fmaf(w, a[j].y, acc.y), fmaf(w, a[j].z, acc.z), fmaf(w, a[j].w, acc.w));
    }
  }
  put_parts(g.out.at(row, kH) + head * kHeadDim, g.out.plane, c,
            make_float4(acc.x / den, acc.y / den, acc.z / den, acc.w / den));
}

// ---- GEMM launches ------------------------------------------------------------------

// Tile shapes of the split GEMM, by the number of rows (96: gate/up only).
enum Shape : int { kRows32K4 = 0, kRows32, kRows64, kRows128, kRows96 };
struct ShapeInfo {
  int rows, cols, wk;
};
constexpr ShapeInfo kShapes[] = {{32, 32, 4}, {32, 64, 2}, {64, 128, 1}, {128, 128, 1}};
// The gate/up GEMM's 64-row shape splits k over two waves, not n.
constexpr ShapeInfo kSwiGLUShapes[] = {{32, 32, 4}, {32, 64, 2}, {64, 64, 2}, {128, 128, 1}, {96, 128, 1}};

// Up to 32 rows the waves split k, so that 32 columns make a workgroup;
// beyond, larger tiles reuse each staged weight for more rows as soon as there
// are enough of them to fill 256 CUs. us at m = 16 / 37 / 128 / 512 / 2048
// (128-row tile: 2048 only), gate/up: 12.2 / 20.4 / 31.4 with 32 rows and four
// k waves, 15.6 / 17.2 / 29.4 with two, 18.1 / 18.7 / 26.9 / 70 with 64 rows,
// 77 (512) / 237 (2048) with 128 rows (64 rows: 267 at 2048).
//
// Gate/up from 193 to 864 rows: 96 x 128 tiles do less per product outside
// the matrix cores, but are few, and a round of 256 that they hardly begin
// costs as much as a full one; so they are taken where they fill more than two
// fifths of their last round. us with 64 / 96 rows (event spans), FP32, F16, BF16:
//   m = 200  43.4 / 40.0    37.6 / 35.2    34.6 / 31.1
//       288  47.3 / 41.8    39.6 / 36.5    36.7 / 32.9
//       512  67.4 / 65.0    59.1 / 56.1    60.4 / 42.9
//       860 110.9 / 99.1    96.5 / 84.9    85.7 / 69.3
// and where not taken
//       300  47.2 / 56.7    40.1 / 49.9    38.0 / 38.2
//       640  78.3 / 95.2    67.4 / 81.5    59.4 / 64.8
//       960 113.5 / 117.2   97.9 / 101.7   90.3 / 75.7
//     1,024 123.9 / 120.4  106.7 / 103.7  104.0 / 78.2
// One rule for the three types: the order of a sum must not depend on the type
// (a BF16 or F16 engine equals an FP32 one with the rounded weights).
Shape gemm_shape(int m, int n, bool swiglu) {
  if (m <= 32) return kRows32K4;
  if (m <= (swiglu ? 64 : 128)) return kRows32;
  if (m > 1024) return kRows128;
  if (!swiglu || m <= 192 || m > 864) return kRows64;
  const int workgroups = (m + 95) / 96 * (n / 64);
  return ((workgroups - 1) % 256 + 1) * 5 > 256 * 2 ? kRows96 : kRows64;
}

template <int RB, int WM, int WN, int WK, typename W, bool kSwiGLU>
void launch_shape(hipStream_t s, const gemm::Args<W> &g) {
  const int mtiles = (g.m + 32 * RB * WM - 1) / (32 * RB * WM);
  const int pairs = g.n / ((kSwiGLU ? 16 : 32) * WN) * g.splits;
  const int grid = (pairs + gemm::kDealXcds - 1) / gemm::kDealXcds * gemm::kDealXcds * mtiles;
  gemm::gemm_split_kernel<RB, WM, WN, WK, W, kSwiGLU><<<grid, gemm::kThreads, 0, s>>>(g, mtiles, pairs);
}

template <typename W>
hipError_t launch_gemm_as(hipStream_t s, gemm::Args<W> g, bool swiglu) {
  const Shape shape = gemm_shape(g.m, g.n, swiglu);
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
      case kRows96: launch_shape<3, 1, 4, 1, W, true>(s, g); break;
      case kRows128: launch_shape<4, 1, 4, 1, W, true>(s, g); break;
    }
  } else {
    switch (shape) {
      case kRows32K4: launch_shape<1, 1, 1, 4, W, false>(s, g); break;
      case kRows32: launch_shape<1, 1, 2, 2, W, false>(s, g); break;
      case kRows64: launch_shape<2, 1, 4, 1, W, false>(s, g); break;
      case kRows96: break;  // not chosen
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
  const ShapeInfo &i = kShapes[gemm_shape(m, n, false)];
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

// Key blocks per workgroup: one until about two workgroups per CU are busy,
// and no more partials than kAttnRecRows rows of records hold.
hipError_t launch_attention_prefill(hipStream_t s, const float *q, int rows, int pos0, const float *k_cache,
                                    const float *v_cache, float *records, const PartRows &out) {
  if (rows <= 0 || pos0 < 0) return hipErrorInvalidValue;
  const int nqb = (rows + kQRows - 1) / kQRows;
  long long units = 0;
  for (int b = 0; b < nqb; ++b) units += (pos0 + std::min(rows, (b + 1) * kQRows) + kKeyBlock - 1) / kKeyBlock;
  const int blocks = (pos0 + rows + kKeyBlock - 1) / kKeyBlock;
  const int most = std::max(1, kAttnRecRows / rows);
  const int per_split = std::max<int>((2 * units + 511) / 512, (blocks + most - 1) / most);
  AttnArgs g{q, k_cache, v_cache, rows, pos0, per_split, (blocks + per_split - 1) / per_split, records, out};
  attention_prefill_kernel<<<dim3(nqb, 2, g.splits), kAttnThreads, 0, s>>>(g);
  if (g.splits > 1) attention_merge_kernel<<<rows, kBlock, 0, s>>>(g);
  return hipGetLastError();
}

}  // namespace qd
