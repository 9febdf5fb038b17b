// Batched decode step for gfx950: up to 16 independent sequences with
// ragged KV lengths advance one token together.
//
// Projections are skinny GEMMs D[seq][row] = sum_k X[seq][k] W[row][k] on
// v_mfma_f32_16x16x4f32: the (up to) 16 sequences are the M dimension and a
// 16-row tile of the weight matrix is N. Lane l of a wave supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and result register r holds
// D[(l / 16) * 4 + r][l % 16]. Each weight is read from HBM once per step for
// the whole batch. The waves of a workgroup split K; both operands reach them
// through LDS rings filled by DMA (split_product); the waves' partial tiles are
// summed in LDS in a fixed order and the 256 tile elements go through the fused
// epilogue (bias, RoPE + KV write, residual add, SiLU gate). The LM head keeps
// the operand rows in LDS and streams the vocabulary past them.
//
// What bounds a step (16 rows): the weights' 1.98 GB would stream in about
// 280 us; a layer's five kernels take 5.1 (QKV), 12.7 (attention, contexts to
// 2,048), 4.7 (O), 10.3 (gate/up) and 7.3 us (down), of which each kernel's
// start, first load and split-K hand-over are most of the three small ones.
// (Kernel trace. The before-and-after figures below are HIP-event spans of
// qd_profile_batch, which hold the gap between two launches too, 2 to 3 us.)
//
// Semantics per sequence are those of the batch-1 step (qd_kernels.hip):
//   RMSNorm                 benchmarks/qwen_stateful_graph_kernel.cpp:665-701
//   QKV + bias, RoPE, KV    benchmarks/qwen_stateful_graph_kernel.cpp:392-552
//   GQA attention           benchmarks/qwen_stateful_graph_kernel.cpp:554-600
//   O / gate-up / down      benchmarks/qwen_stateful_graph_kernel.cpp:158-223,494-515,602-659
//   LM head + top-1         benchmarks/qwen_stateful_graph_kernel.cpp:225-356
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <mutex>

#include "qd_attention.hpp"
#include "qd_batch.hpp"
#include "qd_device.hpp"
#include "qd_device_math.hpp"

namespace qd {
namespace {

using namespace dev;

typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kH = 896;    // hidden = query width
constexpr int kI = 4864;   // MLP intermediate

__device__ __forceinline__ int tile_col() { return lane_id() & 15; }     // N index (weight row)

__device__ __forceinline__ float4 ld4(const float *p) {
  return *reinterpret_cast<const float4 *>(p);
}

__device__ __forceinline__ f4v mfma4(float4 a, float4 b, f4v acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
  return acc;
}

// RMSNorm folded into the GEMM: y = x * inv * g gives W.y = inv * W.(x g).
// The kernel that finishes a hidden row stores x * g for the next norm's gain
// (BatchLaunch::gained) and, per 16-column tile, the sum of the tile's squares
// (BatchLaunch::squares); the GEMMs then load one operand and no gain (whose
// registers kept the gate/up workgroups to two per CU, two rounds of them), and
// their epilogue threads, 16 per sequence, add up the
// row's squares themselves.
__device__ __forceinline__ float row_inv(const BatchLaunch &p, int seq) {
  const float *sq = p.squares + seq * kBatchTiles + (threadIdx.x & 15);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < kBatchTiles / 16; ++j) s += sq[16 * j];
  return rsqrtf(row16_sum(s) / static_cast<float>(kH) + p.eps);
}

// Element v of hidden row seq, column n0 + (t & 15) of tile `tile`, by the
// tile's 256 threads: the row, its gained copy and its share of the squares.
__device__ __forceinline__ void put_hidden(const BatchLaunch &p, int seq, int tile, float v, float gain) {
  const int col = tile * 16 + (threadIdx.x & 15);
  const float ss = row16_sum(v * v);
  if (seq >= p.rows) return;
  p.hidden[seq * kH + col] = v;
  p.gained[seq * kH + col] = v * gain;
  if ((threadIdx.x & 15) == 0) p.squares[seq * kBatchTiles + tile] = ss;
}

// ---- K slices through LDS -------------------------------------------------------
// One wave's product of X[:, k] and W[rows, k] over 32-wide k slices
// [s0, s1), both operands through the wave's own ring of kRing LDS stages
// (2 KiB of X, 2 KiB of W each), filled by global -> LDS DMA. A DMA moves
// whole 128-byte lines (8 rows of a slice), where a load into the operand
// layout (16 rows x 64 bytes) takes every line in two halves; and no registers
// wait for memory. The ring is the wave's own, so no barrier. Against operand
// loads into registers, 16 rows, per layer: gate/up 19.1 -> 12.8 us, down
// 12 -> 10, QKV 9.8 -> 8.0. (Rings of 2 or 4 stages: 1161 and 1173 us a step
// against 1162; K = 896 in 3 or 4 splits and down in 6: 1178.)
// Rows are 32 floats, 16-byte slot p holding piece p ^ ((row / 2) % 8): the 16
// rows' reads of one piece fall on distinct banks.
constexpr int kSlice = 32, kRing = 3, kStageFloats = 2 * 16 * kSlice, kRingFloats = kRing * kStageFloats;
typedef __attribute__((address_space(3))) void ring_lds_void;
// kOnce: bytes that no other workgroup reads (weights), not to be kept in L2
// (LM head at 16 rows 113 -> 106 us).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is reserved: set before each use, never saved
template <bool kOnce>
__device__ __forceinline__ void ring_dma(const float *src, uint32_t lds) {
  if constexpr (kOnce)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(src)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
template <int n>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}
// The DMA source of this lane for instruction i of a 16-row, 32-column slice:
// its 16-byte piece of row 8 i + lane / 8.
__device__ __forceinline__ int ring_row(int i) { return 8 * i + (lane_id() >> 3); }
__device__ __forceinline__ int ring_piece(int row) { return 4 * ((lane_id() & 7) ^ ((row >> 1) & 7)); }
__device__ __forceinline__ uint32_t ring_address(const float *ring) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>((ring_lds_void *)ring))));
}
// Operand float4s of k's 4 (l / 16) .. + 3 and 16 further on, row l % 16 of a slice.
__device__ __forceinline__ void ring_read(const float *slice, float4 &a, float4 &b) {
  const int row = lane_id() & 15, sw = (row >> 1) & 7, quad = lane_id() >> 4;
  const float4 *r = reinterpret_cast<const float4 *>(slice) + row * 8;
  a = r[quad ^ sw];
  b = r[(4 + quad) ^ sw];
}

// This wave's part of X . W^T over K floats per row (X row i at x + i K, W row
// j at wrow(j)), K dealt in slices to the waves of kSplits workgroups.
template <int K, int kSplits, typename WRow>
__device__ __forceinline__ f4v split_product(float (*rings)[kRingFloats], const float *x, WRow wrow) {
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  constexpr int kWaves = kWavesPerBlock * kSplits, kSlices = K / kSlice;
  const int part = blockIdx.y * kWavesPerBlock + w;
  const int s0 = part * kSlices / kWaves, n = (part + 1) * kSlices / kWaves - s0;
  const float *ring = rings[w];
  const uint32_t base = ring_address(ring);
  const float *src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = ring_row(i & 1);
    src[i] = (i < 2 ? x + row * K : wrow(row)) + s0 * kSlice + ring_piece(row);
  }
  auto fetch = [&](int stage) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t dst = base + stage * kStageFloats * 4 + i * 1024;
      if (i < 2)
        ring_dma<false>(src[i], dst);
      else
        ring_dma<true>(src[i], dst);
      src[i] += kSlice;
    }
  };
#pragma unroll
  for (int d = 0; d < kRing; ++d)
    if (d < n) fetch(d);
  f4v acc = {0.f, 0.f, 0.f, 0.f};
  int stage = 0;
  for (int s = 0; s < n; ++s) {
    // Stage s has landed once at most the later stages' DMAs, four each, are
    // outstanding.
    static_assert(kRing == 3, "two later stages at most");
    if (n - 1 - s >= 2)
      ring_wait<8>();
    else if (n - 1 - s == 1)
      ring_wait<4>();
    else
      ring_wait<0>();
    float4 x0, x1, w0, w1;
    ring_read(ring + stage * kStageFloats, x0, x1);
    ring_read(ring + stage * kStageFloats + 16 * kSlice, w0, w1);
    acc = mfma4(x0, w0, acc);
    acc = mfma4(x1, w1, acc);
    // The operands are in registers: the stage can be filled again.
    if (s + kRing < n) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      fetch(stage);
    }
    stage = stage + 1 == kRing ? 0 : stage + 1;
  }
  return acc;
}

// Sums the waves' partial tiles: red is [waves][4][64]; thread t < 256
// returns element (register t / 64, lane t % 64), i.e. sequence
// ((t % 64) / 16) * 4 + t / 64 and tile column t % 16. Starts and ends
// with a workgroup barrier.
template <int kWaves>
__device__ __forceinline__ float tile_reduce(f4v acc, float (*red)[4][kWave]) {
  const int w = wave_id(), l = lane_id();
#pragma unroll
  for (int r = 0; r < 4; ++r) red[w][r][l] = acc[r];
  __syncthreads();
  float v = 0.f;
  const int t = threadIdx.x;
  if (t < 4 * kWave) {
#pragma unroll
    for (int u = 0; u < kWaves; ++u) v += red[u][t >> 6][t & 63];
  }
  __syncthreads();
  return v;
}

__device__ __forceinline__ int tile_seq(int t) { return ((t & 63) >> 4) * 4 + (t >> 6); }

// Waits until this thread's vector memory operations have completed (gfx9
// s_waitcnt encoding: vmcnt 0, expcnt and lgkmcnt not waited on).
__device__ __forceinline__ void wait_vm_stores() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Split-K over workgroups: workgroup blockIdx.y of kSplits deposits its
// partial tile (thread t < 256 holds element t); the last workgroup of the
// tile to arrive sums the deposits in split order (deterministic) into v,
// resets the tile's counter and returns true. Other workgroups return false.
// Deposits use device-scope (sc1) stores and loads, which are coherent across
// the XCDs' L2s without an L2 writeback or invalidate; each depositing thread
// waits for its stores to complete before the workgroup's arrival is counted.
constexpr int kSplitRec = 256;
template <int kSplits>
__device__ bool split_gather(float &v, float *__restrict__ ws, uint32_t *cnt, int tile) {
  __shared__ uint32_t last;
  const int t = threadIdx.x;
  if (kSplits == 1) return true;
  const Coherent dep(ws + static_cast<size_t>(tile) * kSplits * kSplitRec,
                     static_cast<uint32_t>(kSplits * kSplitRec * sizeof(float)));
  dep.st(blockIdx.y * kSplitRec + t, v);
  wait_vm_stores();
  __syncthreads();
  if (t == 0) last = atomicAdd(cnt + tile, 1u) == static_cast<uint32_t>(kSplits - 1);
  __syncthreads();
  if (!last) return false;
  // All deposits are requested before any is summed (one round trip).
  float pv[kSplits];
#pragma unroll
  for (int s = 0; s < kSplits; ++s) pv[s] = dep.ld(s * kSplitRec + t);
  float sum = 0.f;
#pragma unroll
  for (int s = 0; s < kSplits; ++s) sum += pv[s];
  v = sum;
  if (t == 0) cnt[tile] = 0u;
  return true;
}

// Counter regions of BatchLaunch::counters.
constexpr int kCntQkv = 0, kCntO = 128, kCntDown = 256, kCntAttn = 512;

__device__ __forceinline__ float *kv_rows(float *cache, uint32_t slot, int layer, int layers,
                                          int capacity, int kv_dim) {
  return cache + (static_cast<size_t>(slot) * layers + layer) * capacity * kv_dim;
}

// Rows of a K or V cache through a buffer descriptor that ends with the last
// one wanted: a load past it returns zeros and touches no memory.
struct KvRows {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ KvRows(const float *base, uint32_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, static_cast<int>(bytes), kRsrcWord3)) {}
  __device__ __forceinline__ float ld(uint32_t i) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, i * 4u, 0, 0));
  }
  __device__ __forceinline__ float4 ld4(uint32_t i) const {
    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, i * 4u, 0, 0));
    return make_float4(v[0], v[1], v[2], v[3]);
  }
};

// ---- kernels --------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void batch_embed_kernel(BatchLaunch p, const float *__restrict__ emb,
                                                             const float *__restrict__ gain, int vocab) {
  const int b = blockIdx.x;
  const uint32_t tok = p.token[b];
  if (tok >= static_cast<uint32_t>(vocab)) return;
  const float *src = emb + static_cast<size_t>(tok) * kH;
  for (int tile = threadIdx.x >> 4; tile < kH / 16; tile += kBlock / 16) {
    const int col = tile * 16 + (threadIdx.x & 15);
    put_hidden(p, b, tile, src[col], gain[col]);
  }
}

// Attention RMSNorm + packed QKV + bias + RoPE + KV-cache write. Tile
// blockIdx.x holds, for head T / 4 and i0 = 8 * (T % 4), the rows
// head*64 + i0 + j and head*64 + 32 + i0 + j (j < 8) as tile columns j and
// j + 8: the rotate-half partners sit in lanes l and l ^ 8. Heads [0, nq)
// are queries, then nkv keys, then nkv values (not rotated). K = 896 is
// split over kQkvSplit workgroups of four waves (two: 144 workgroups instead
// of 72).
constexpr int kQkvSplit = 2;
__global__ __launch_bounds__(kBlock) void batch_qkv_kernel(BatchLaunch p, const float *__restrict__ wqkv,
                                                           const float *__restrict__ bqkv, int layer) {
  __shared__ __attribute__((aligned(16))) float ring[kWavesPerBlock][kRingFloats];
  __shared__ float red[kWavesPerBlock][4][kWave];
  const int tile = blockIdx.x;
  const int head = tile >> 2;
  const int i0 = (tile & 3) * 8;
  // Epilogue element of this thread: its bias and rotation are requested
  // with the weights.
  const int t = threadIdx.x;
  const int seq = tile_seq(t);
  const int jt = t & 15;
  const int i = i0 + (jt & 7);
  const int row = head * kHeadDim + (jt < 8 ? i : kRotary + i);
  const int pos = static_cast<int>(p.pos[min(seq, p.rows - 1)]);
  const float bias = bqkv[row];
  const float c = p.rope_cos[pos * kRotary + i];
  const float s = p.rope_sin[pos * kRotary + i];
  const float inv = row_inv(p, seq);
  const f4v acc = split_product<kH, kQkvSplit>(ring, p.gained, [&](int j) {
    return wqkv + static_cast<size_t>(head * kHeadDim + (j < 8 ? i0 + j : kRotary + i0 + j - 8)) * kH;
  });
  float v = tile_reduce<kWavesPerBlock>(acc, red);
  if (!split_gather<kQkvSplit>(v, p.split, p.counters + kCntQkv, tile)) return;
  // Epilogue over the 256 tile elements.
  v = v * inv + bias;
  const float other = __shfl_xor(v, 8, kWave);
  if (seq >= p.rows) return;
  const uint32_t slot = p.slot[seq];
  const int kv_dim = p.nkv * kHeadDim;
  const int d = row - head * kHeadDim;
  if (head < p.nq + p.nkv) {
    // (a, b) = (row i, row i + 32): a' = a c - b s, b' = b c + a s.
    const float out = jt < 8 ? v * c - other * s : v * c + other * s;
    if (head < p.nq) {
      p.q[seq * (p.nq * kHeadDim) + row] = out;
    } else {
      float *kc = kv_rows(p.k_cache, slot, layer, p.layers, p.capacity, kv_dim);
      kc[static_cast<size_t>(pos) * kv_dim + (head - p.nq) * kHeadDim + d] = out;
    }
  } else {
    float *vc = kv_rows(p.v_cache, slot, layer, p.layers, p.capacity, kv_dim);
    vc[static_cast<size_t>(pos) * kv_dim + (head - p.nq - p.nkv) * kHeadDim + d] = v;
  }
}

// GQA decode attention on the matrix cores: workgroup (chunk, KV group g,
// batch row b) serves all query heads of the group (up to 16), so every K/V
// row of the chunk is read once. Waves take 16-position tiles (wave w: tile
// w of each 128-position pass). Per tile:
//   S[head][pos] = (Q / 8) . K^T    16x16x4 MFMAs, lane l supplies
//                                   Q[head l%16] and K[pos l%16] at dims
//                                   16 s + 4 (l/16) + c (float4 loads)
//   online softmax per head row     (S register r of lane l is head
//                                   4 (l/16) + r, position l%16: row
//                                   reductions over the 16-lane DPP rows)
//   O[head][d] += P . V             P goes through the wave's LDS to become
//                                   the A operand; V is loaded as B operands.
// The wave partials are merged into one record (m, l, acc[64]) per head; the
// last chunk of (b, g) to finish merges all chunks (the same merge as
// attn_merge) into attn[b][h*64 + d]. Q is scaled by kScoreScaleLog2 =
// log2(e) / sqrt(64), so scores and maxima are in base-2 units and every
// softmax exponential is one v_exp_f32 (2^x).
//
// Bound by latency (a layer's K/V rows of 16 contexts to 2,048, 19 MB, stream
// in 3 us): one round trip for the K and V of a wave's only tile, which are
// requested before anything else, then the record and counter round trips.
// Per layer 18.0 -> 14.8 us at 16 rows (five rows, contexts to 300: 11.3 ->
// 10.7) against chunks of four waves that passed over up to three tiles each,
// V through LDS.
constexpr int kAttnWaves = 8, kAttnThreads = kAttnWaves * kWave, kAttnTileRows = 16;
struct GqaLds {
  float ps[kAttnWaves][16][17];   // P tile [head][pos]
  float wm[kAttnWaves][16];
  float wl[kAttnWaves][16];
  float wo[kAttnWaves][16][65];   // wave partial O [head][dim]
};

// Positions per chunk: one tile per wave while kAttnMaxChunks such chunks hold
// the context (2,048 positions), then the fewest tiles that hold it.
__device__ __forceinline__ int batch_chunk_len(int length) {
  return max(attn_chunk_len(length, kAttnMaxChunks, kAttnTileRows), kAttnWaves * kAttnTileRows);
}

__global__ __launch_bounds__(kAttnThreads, 4) void batch_attn_kernel(BatchLaunch p, int layer) {
  __shared__ GqaLds sh;
  __shared__ uint32_t last;
  const int b = blockIdx.z, g = blockIdx.y, chunk = blockIdx.x;
  const uint32_t slot = p.slot[b];
  const int position = static_cast<int>(p.pos[b]);
  const int length = position + 1;
  const int chunk_len = batch_chunk_len(length);
  const int chunks = (length + chunk_len - 1) / chunk_len;
  if (chunk >= chunks) return;
  const int begin = chunk * chunk_len;
  const int end = min(length, begin + chunk_len);
  const int group = p.nq / p.nkv;
  const int kv_dim = p.nkv * kHeadDim;
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), col = tile_col(), quad = lane_id() >> 4;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);

  // The chunk's K and V rows of the group: the descriptor ends after row
  // end - 1, and rows past it read as zeros.
  const size_t first = static_cast<size_t>(begin) * kv_dim + g * kHeadDim;
  const uint32_t bytes = ((end - begin) * kv_dim - g * kHeadDim) * sizeof(float);
  const KvRows kr(kv_rows(p.k_cache, slot, layer, p.layers, p.capacity, kv_dim) + first, bytes);
  const KvRows vr(kv_rows(p.v_cache, slot, layer, p.layers, p.capacity, kv_dim) + first, bytes);
  float4 kc[4];
  float vc[4][4];
  auto load_k = [&](int row) {
#pragma unroll
    for (int s = 0; s < 4; ++s) kc[s] = kr.ld4((row + col) * kv_dim + 16 * s + 4 * quad);
  };
  auto load_v = [&](int row) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n = 0; n < 4; ++n) vc[s][n] = vr.ld((row + 4 * s + quad) * kv_dim + 16 * n + col);
  };
  const int rows = end - begin;
  int row = kAttnTileRows * w;
  load_k(row);
  load_v(row);
  float4 qa[4];
  if (col < group) {
    const float *qr = p.q + b * (p.nq * kHeadDim) + (g * group + col) * kHeadDim + 4 * quad;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float4 v = ld4(qr + 16 * s);
      qa[s] = make_float4(v.x * kScoreScaleLog2, v.y * kScoreScaleLog2, v.z * kScoreScaleLog2,
                          v.w * kScoreScaleLog2);
    }
  } else {
#pragma unroll
    for (int s = 0; s < 4; ++s) qa[s] = zero;
  }

  float m[4], lsum[4];
  f4v o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = -INFINITY;
    lsum[r] = 0.f;
    o[r] = f4v{0.f, 0.f, 0.f, 0.f};
  }
  for (; row < rows; row += kAttnTileRows * kAttnWaves) {
    const bool more = row + kAttnTileRows * kAttnWaves < rows;
    f4v sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) sacc = mfma4(qa[s], kc[s], sacc);
    if (more) load_k(row + kAttnTileRows * kAttnWaves);
    const bool valid = row + col < rows;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float sv = valid ? sacc[r] : -INFINITY;
      const float mn = fmaxf(m[r], row16_max(sv));
      const float pv = mn == -INFINITY ? 0.f : exp2_fast(sv - mn);
      const float corr = mn == -INFINITY ? 1.f : exp2_fast(m[r] - mn);
      lsum[r] = fmaf(lsum[r], corr, row16_sum(pv));
      m[r] = mn;
#pragma unroll
      for (int n = 0; n < 4; ++n) o[n][r] *= corr;
      sh.ps[w][4 * quad + r][col] = pv;
    }
    // The wave's own LDS tile: LDS operations of a wave complete in order.
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float a = sh.ps[w][col][4 * s + quad];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        o[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vc[s][n], o[n], 0, 0, 0);
    }
    if (more) load_v(row + kAttnTileRows * kAttnWaves);
  }
  // Wave partials -> one record per head of the group.
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (col == 0) {
      sh.wm[w][4 * quad + r] = m[r];
      sh.wl[w][4 * quad + r] = lsum[r];
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) sh.wo[w][4 * quad + r][16 * n + col] = o[n][r];
  }
  __syncthreads();
  const Coherent recs(p.part + (static_cast<size_t>(b) * p.nq + g * group) * kAttnMaxChunks * kPartStride,
                      group * kAttnMaxChunks * kPartStride * sizeof(float));
  for (int i = threadIdx.x; i < group * kHeadDim; i += kAttnThreads) {
    const int h = i / kHeadDim, d = i % kHeadDim;
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < kAttnWaves; ++v) mx = fmaxf(mx, sh.wm[v][h]);
    float lt = 0.f, a = 0.f;
#pragma unroll
    for (int v = 0; v < kAttnWaves; ++v) {
      const float f = sh.wm[v][h] == -INFINITY ? 0.f : exp2_fast(sh.wm[v][h] - mx);
      lt = fmaf(f, sh.wl[v][h], lt);
      a = fmaf(f, sh.wo[v][h][d], a);
    }
    const uint32_t rec = (h * kAttnMaxChunks + chunk) * kPartStride;
    recs.st(rec + 2 + d, a);
    if (d == 0) {
      recs.st(rec, mx);
      recs.st(rec + 1, lt);
    }
  }
  wait_vm_stores();
  __syncthreads();
  uint32_t *cnt = p.counters + kCntAttn + b * p.nkv + g;
  if (threadIdx.x == 0) last = atomicAdd(cnt, 1u) == static_cast<uint32_t>(chunks - 1);
  __syncthreads();
  if (!last) return;
  for (int i = threadIdx.x; i < group * kHeadDim; i += kAttnThreads) {
    const int h = i / kHeadDim, d = i % kHeadDim;
    const uint32_t head_rec = h * kAttnMaxChunks * kPartStride;
    // Every chunk's (m, l, acc_d) is requested before any is used.
    float cm[kAttnMaxChunks], cl[kAttnMaxChunks], ca[kAttnMaxChunks];
#pragma unroll
    for (int c = 0; c < kAttnMaxChunks; ++c) {
      const uint32_t rec = head_rec + c * kPartStride;
      const bool in = c < chunks;
      cm[c] = in ? recs.ld(rec) : -INFINITY;
      cl[c] = in ? recs.ld(rec + 1) : 0.f;
      ca[c] = in ? recs.ld(rec + 2 + d) : 0.f;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < kAttnMaxChunks; ++c) mx = fmaxf(mx, cm[c]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int c = 0; c < kAttnMaxChunks; ++c) {
      const float f = c < chunks ? exp2_fast(cm[c] - mx) : 0.f;
      den = fmaf(f, cl[c], den);
      num = fmaf(f, ca[c], num);
    }
    p.attn[b * (p.nq * kHeadDim) + (g * group + h) * kHeadDim + d] = num / den;
  }
  if (threadIdx.x == 0) *cnt = 0u;
}

// hidden[b][row] += Wo[row] . attn[b] for the 16 rows of tile blockIdx.x;
// K = 896 split over kOSplit workgroups (two: 112 workgroups instead of 56).
constexpr int kOSplit = 2;
__global__ __launch_bounds__(kBlock) void batch_oproj_kernel(BatchLaunch p, const float *__restrict__ wo,
                                                             const float *__restrict__ next_gain) {
  __shared__ __attribute__((aligned(16))) float ring[kWavesPerBlock][kRingFloats];
  __shared__ float red[kWavesPerBlock][4][kWave];
  const int tile = blockIdx.x, n0 = tile * 16;
  const f4v acc = split_product<kH, kOSplit>(ring, p.attn, [&](int j) { return wo + static_cast<size_t>(n0 + j) * kH; });
  float v = tile_reduce<kWavesPerBlock>(acc, red);
  const int t = threadIdx.x, seq = tile_seq(t);
  const float gain = next_gain[n0 + (t & 15)];
  if (!split_gather<kOSplit>(v, p.split, p.counters + kCntO, tile)) return;
  put_hidden(p, seq, tile, p.hidden[seq * kH + n0 + (t & 15)] + v, gain);
}

// MLP RMSNorm + gate/up + SiLU: act[b][row] = silu(g) * u. Tile blockIdx.x
// covers rows n0 .. n0 + 7 of the activation: tile column j < 8 is gate row
// n0 + j and column j + 8 the up row n0 + j, and the 608 tiles (of 57 KB each) spread evenly over the CUs. The up
// sum crosses to its gate lane (column j + 8 -> j) by a lane exchange.
__global__ __launch_bounds__(kBlock) void batch_gateup_kernel(BatchLaunch p, const float *__restrict__ wg,
                                                              const float *__restrict__ wu) {
  __shared__ __attribute__((aligned(16))) float ring[kWavesPerBlock][kRingFloats];
  __shared__ float red[kWavesPerBlock][4][kWave];
  const int n0 = blockIdx.x * 8;
  const int t = threadIdx.x;
  const int seq = tile_seq(t);
  const float inv = row_inv(p, seq);
  const f4v acc = split_product<kH, 1>(
      ring, p.gained, [&](int j) { return (j < 8 ? wg : wu) + static_cast<size_t>(n0 + (j & 7)) * kH; });
  const float v = tile_reduce<kWavesPerBlock>(acc, red);
  // Thread t < 256 holds (sequence tile_seq(t), column t & 15); its partner
  // column t ^ 8 sits in lane (t ^ 8) of the same wave.
  const float other = __shfl_xor(v, 8, kWave);
  if ((t & 15) < 8 && seq < p.rows) {
    const float g = v * inv, u = other * inv;
    p.act[seq * kI + n0 + (t & 7)] = g / (1.f + expf(-g)) * u;
  }
}

// hidden[b][row] += Wd[row] . act[b]; K = 4864 split over kDownSplit
// workgroups of four waves.
constexpr int kDownSplit = 4;
__global__ __launch_bounds__(kBlock) void batch_down_kernel(BatchLaunch p, const float *__restrict__ wd,
                                                            const float *__restrict__ next_gain) {
  __shared__ __attribute__((aligned(16))) float ring[kWavesPerBlock][kRingFloats];
  __shared__ float red[kWavesPerBlock][4][kWave];
  const int tile = blockIdx.x, n0 = tile * 16;
  const f4v acc = split_product<kI, kDownSplit>(ring, p.act, [&](int j) { return wd + static_cast<size_t>(n0 + j) * kI; });
  float v = tile_reduce<kWavesPerBlock>(acc, red);
  const int t = threadIdx.x, seq = tile_seq(t);
  const float gain = next_gain[n0 + (t & 15)];
  if (!split_gather<kDownSplit>(v, p.split, p.counters + kCntDown, tile)) return;
  put_hidden(p, seq, tile, p.hidden[seq * kH + n0 + (t & 15)] + v, gain);
}

// Final RMSNorm + tied LM head + per-workgroup top-1 of every batch row. One
// workgroup of eight waves per CU: the gain-scaled rows sit in LDS (57 KiB) as
// the matrix operand of every wave; a wave streams whole vocabulary tiles of 16
// rows on its own through a ring of kLmRing LDS slices (2 KiB each), with no
// barrier and no sum across waves. 16 rows: 106 us for 545 MB (5.1 TB/s; a plain
// copy reaches 5.2), against 125 with four-way split tiles through registers.
constexpr int kLmWaves = 8, kLmThreads = kLmWaves * kWave;
constexpr int kLmRing = 6, kLmSlice = 16 * kSlice;  // floats of a slice
constexpr int kLmRow = kH + 4;  // LDS row stride: the 16 rows' reads on distinct banks
__global__ __launch_bounds__(kLmThreads) void batch_lmhead_kernel(BatchLaunch p, BatchTail tl) {
  __shared__ __attribute__((aligned(16))) float xs[16 * kLmRow];
  __shared__ __attribute__((aligned(16))) float rings[kLmWaves][kLmRing * kLmSlice];
  __shared__ float invs[16];
  __shared__ float wv[kLmWaves][16];
  __shared__ uint32_t wi[kLmWaves][16];
  const int tiles = (tl.vocab + 15) / 16, stride = gridDim.x * kLmWaves;
  const int n = tile_col(), lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id()), lg = lane >> 4;
  for (int i = threadIdx.x; i < 16 * kH / 4; i += kLmThreads) {
    const int b = i / (kH / 4), c = i % (kH / 4);
    *reinterpret_cast<float4 *>(xs + b * kLmRow + 4 * c) =
        b < p.rows ? ld4(p.gained + b * kH + 4 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (threadIdx.x < 256) {
    const float inv = row_inv(p, tile_seq(threadIdx.x));
    if ((threadIdx.x & 15) == 0) invs[tile_seq(threadIdx.x)] = inv;
  }
  __syncthreads();
  // This lane's sequences 4 lg + r: scale, logits row, running top-1.
  float inv[4], best[4];
  uint32_t best_i[4];
  float *out[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int seq = 4 * lg + r;
    inv[r] = invs[seq];
    best[r] = -INFINITY;
    best_i[r] = UINT32_MAX;
    out[r] = seq < p.rows ? tl.logits + static_cast<size_t>(p.slot[seq]) * tl.vocab : nullptr;
  }
  const float *ring = rings[w];
  const uint32_t base = ring_address(ring);
  const float *x = xs + n * kLmRow + 4 * lg;
  constexpr int kSlices = kH / kSlice;  // 28 per tile
  int tile = blockIdx.x + w * gridDim.x;
  // The slices to fetch, kLmRing ahead of the one multiplied: next_slice of
  // next_tile. Past the last tile the last one is fetched again, so that every
  // slice is followed by the same number of DMAs.
  int next_tile = tile, next_slice = 0;
  const float *src[2];
  auto aim = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = ring_row(i);
      src[i] = tl.head + static_cast<size_t>(min(next_tile * 16 + row, tl.vocab - 1)) * kH + ring_piece(row);
    }
  };
  auto fetch = [&](int stage) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ring_dma<true>(src[i], base + (stage * kLmSlice + i * 256) * 4);
      src[i] += kSlice;
    }
    if (++next_slice == kSlices) {
      next_slice = 0;
      next_tile = next_tile + stride < tiles ? next_tile + stride : next_tile;
      aim();
    }
  };
  int stage = 0;
  if (tile < tiles) {
    aim();
#pragma unroll
    for (int d = 0; d < kLmRing; ++d) fetch(d);
  }
  for (; tile < tiles; tile += stride) {
    f4v acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < kSlices; ++s) {
      // (The logits' stores count too: a wait that finds them outstanding
      // only waits for more.)
      ring_wait<2 * (kLmRing - 1)>();
      float4 w0, w1;
      ring_read(ring + stage * kLmSlice, w0, w1);
      const float4 x0 = ld4(x + s * kSlice), x1 = ld4(x + s * kSlice + 16);
      acc = mfma4(x0, w0, acc);
      acc = mfma4(x1, w1, acc);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      fetch(stage);
      stage = stage + 1 == kLmRing ? 0 : stage + 1;
    }
    const int row = tile * 16 + n;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = acc[r] * inv[r];
      if (out[r] && row < tl.vocab) {
        out[r][row] = v;
        if (better(v, static_cast<uint32_t>(row), best[r], best_i[r])) {
          best[r] = v;
          best_i[r] = static_cast<uint32_t>(row);
        }
      }
    }
  }
  ring_wait<0>();  // the ring's last fetches land before the workgroup goes
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const float ov = __shfl_xor(best[r], o, kWave);
      const uint32_t oi = __shfl_xor(best_i[r], o, kWave);
      if (better(ov, oi, best[r], best_i[r])) {
        best[r] = ov;
        best_i[r] = oi;
      }
    }
    if (n == 0) {
      wv[w][4 * lg + r] = best[r];
      wi[w][4 * lg + r] = best_i[r];
    }
  }
  __syncthreads();
  if (threadIdx.x >= p.rows) return;
  float top = wv[0][threadIdx.x];
  uint32_t top_i = wi[0][threadIdx.x];
#pragma unroll
  for (int u = 1; u < kLmWaves; ++u)
    if (better(wv[u][threadIdx.x], wi[u][threadIdx.x], top, top_i)) {
      top = wv[u][threadIdx.x];
      top_i = wi[u][threadIdx.x];
    }
  tl.part_val[threadIdx.x * kBatchLmParts + blockIdx.x] = top;
  tl.part_idx[threadIdx.x * kBatchLmParts + blockIdx.x] = top_i;
}

// Per batch row: reduces the top-1 partials and writes the slot's state as
// a step leaves it (token sampled, position advanced), as
// argmax_finalize_kernel does for one sequence.
__global__ __launch_bounds__(kBlock) void batch_argmax_kernel(BatchLaunch p, BatchTail tl) {
  __shared__ float bv[kWavesPerBlock];
  __shared__ uint32_t bi[kWavesPerBlock];
  const int b = blockIdx.x;
  float best = -INFINITY;
  uint32_t best_i = UINT32_MAX;
  for (int i = threadIdx.x; i < kBatchLmParts; i += kBlock) {
    const float v = tl.part_val[b * kBatchLmParts + i];
    const uint32_t x = tl.part_idx[b * kBatchLmParts + i];
    if (better(v, x, best, best_i)) {
      best = v;
      best_i = x;
    }
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, kWave);
    const uint32_t oi = __shfl_xor(best_i, o, kWave);
    if (better(ov, oi, best, best_i)) {
      best = ov;
      best_i = oi;
    }
  }
  if (lane_id() == 0) {
    bv[wave_id()] = best;
    bi[wave_id()] = best_i;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kWavesPerBlock; ++w) {
    if (better(bv[w], bi[w], best, best_i)) {
      best = bv[w];
      best_i = bi[w];
    }
  }
  SeqState st{};
  st.position = p.pos[b] + 1;
  st.token = best_i;
  st.eos = UINT32_MAX;
  st.top_logit = best;
  st.mode = kModeStep;
  // Every logit NaN: nothing can be fed back (stop reason 0).
  st.stopped = best_i == UINT32_MAX ? 1u : 0u;
  p.states[p.slot[b]] = st;
  tl.out_token[b] = best_i;
  tl.out_top[b] = best;
}

struct Scope {
  Marker *m;
  int id;
  Scope(Marker *marker, int kernel) : m(marker), id(kernel) {
    if (m) m->before(id);
  }
  ~Scope() {
    if (m) m->after(id);
  }
};

__global__ void clear_counters_kernel(uint32_t *__restrict__ counters, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) counters[i] = 0u;
}

// The static batch workspace: one copy per GPU the library runs on. Host
// code never passes this name to a kernel (on the host it is a stand-in,
// not a device address); it uses the per-device address batch_scratch()
// obtains from hipGetSymbolAddress.
__device__ __align__(256) static unsigned char scratch[kBatchScratchBytes];

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxScratchDevices] = {};

size_t round256(size_t bytes) { return (bytes + 255) / 256 * 256; }

}  // namespace

size_t batch_workspace_bytes(int nq) {
  const size_t r = kBatchRows, qd = size_t(nq) * kHeadDim;
  return 2 * round256(r * kH * 4) + round256(r * kBatchTiles * 4) + 2 * round256(r * qd * 4) + round256(r * kI * 4) +
         round256(r * nq * kAttnMaxChunks * kPartStride * 4) + round256(size_t(kBatchSplitFloats) * 4) +
         round256(size_t(kBatchCounters) * 4) + 2 * round256(r * kBatchLmParts * 4) + 2 * round256(r * 4);
}

BatchWorkspace carve_batch_workspace(void *base, int nq) {
  unsigned char *p = static_cast<unsigned char *>(base);
  auto take = [&](size_t bytes) {
    void *r = p;
    p += round256(bytes);
    return r;
  };
  const size_t r = kBatchRows, qd = size_t(nq) * kHeadDim;
  BatchWorkspace w{};
  w.hidden = static_cast<float *>(take(r * kH * 4));
  w.gained = static_cast<float *>(take(r * kH * 4));
  w.squares = static_cast<float *>(take(r * kBatchTiles * 4));
  w.q = static_cast<float *>(take(r * qd * 4));
  w.attn = static_cast<float *>(take(r * qd * 4));
  w.act = static_cast<float *>(take(r * kI * 4));
  w.part = static_cast<float *>(take(r * nq * kAttnMaxChunks * kPartStride * 4));
  w.split = static_cast<float *>(take(size_t(kBatchSplitFloats) * 4));
  w.counters = static_cast<uint32_t *>(take(size_t(kBatchCounters) * 4));
  w.part_val = static_cast<float *>(take(r * kBatchLmParts * 4));
  w.part_idx = static_cast<uint32_t *>(take(r * kBatchLmParts * 4));
  w.out_token = static_cast<uint32_t *>(take(r * 4));
  w.out_top = static_cast<float *>(take(r * 4));
  return w;
}

static_assert(kH / kHeadDim == 14, "the batched kernels take 14 query heads");

void *batch_scratch(int device, hipError_t *err) {
  *err = hipSuccess;
  if (device < 0 || device >= kMaxScratchDevices) {
    *err = hipErrorInvalidDevice;
    return nullptr;
  }
  if (batch_workspace_bytes(kH / kHeadDim) > kBatchScratchBytes) {
    *err = hipErrorInvalidValue;
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      *err = e != hipSuccess ? e : hipErrorInvalidSymbol;
      return nullptr;
    }
    g_scratch_ptr[device] = p;
  }
  return g_scratch_ptr[device];
}

std::mutex &batch_scratch_lock(int device) {
  static std::mutex locks[kMaxScratchDevices];
  return locks[device >= 0 && device < kMaxScratchDevices ? device : 0];
}

hipError_t launch_batch_clear_counters(hipStream_t s, uint32_t *counters) {
  clear_counters_kernel<<<(kBatchCounters + kBlock - 1) / kBlock, kBlock, 0, s>>>(counters, kBatchCounters);
  return hipGetLastError();
}

const char *batch_kernel_name(int id) {
  static const char *const names[kBatchKernelCount] = {
      "batch_embed_kernel",  "batch_qkv_kernel",    "batch_attn_kernel",
      "batch_oproj_kernel",  "batch_gateup_kernel",
      "batch_down_kernel",   "batch_lmhead_kernel", "batch_argmax_kernel"};
  return id >= 0 && id < kBatchKernelCount ? names[id] : "unknown";
}

static bool batch_shape_ok(const BatchLaunch &b) {
  return b.rows >= 1 && b.rows <= kBatchRows && b.nkv > 0 && b.nq % b.nkv == 0 &&
         b.nq * kHeadDim == kH && b.nq / b.nkv <= kMaxGroup && kBatchRows * b.nq <= kBatchCounters - kCntAttn &&
         (b.nq + 2 * b.nkv) * 4 <= kCntO - kCntQkv;
}

hipError_t launch_batch_embed(hipStream_t s, const BatchLaunch &b, const float *embed, const float *first_gain,
                              int vocab, Marker *m) {
  if (!batch_shape_ok(b)) return hipErrorInvalidValue;
  for (int i = 0; i < b.rows; ++i)
    if (b.pos[i] >= static_cast<uint32_t>(b.capacity) || b.token[i] >= static_cast<uint32_t>(vocab))
      return hipErrorInvalidValue;
  Scope scope(m, kBEmbed);
  batch_embed_kernel<<<b.rows, kBlock, 0, s>>>(b, embed, first_gain, vocab);
  return hipGetLastError();
}

hipError_t launch_batch_layer(hipStream_t s, const BatchLaunch &b, const LayerPtrs &w, int layer,
                              const float *next_gain, Marker *m) {
  if (!batch_shape_ok(b)) return hipErrorInvalidValue;
  {
    Scope scope(m, kBQkvRope);
    batch_qkv_kernel<<<dim3((b.nq + 2 * b.nkv) * 4, kQkvSplit), kBlock, 0, s>>>(
        b, w.wqkv, w.bqkv, layer);
  }
  {
    Scope scope(m, kBAttn);
    batch_attn_kernel<<<dim3(kAttnMaxChunks, b.nkv, b.rows), kAttnThreads, 0, s>>>(b, layer);
  }
  {
    Scope scope(m, kBOproj);
    batch_oproj_kernel<<<dim3(kH / 16, kOSplit), kBlock, 0, s>>>(b, w.wo, w.mlp_norm);
  }
  {
    Scope scope(m, kBGateUp);
    batch_gateup_kernel<<<kI / 8, kBlock, 0, s>>>(b, w.wg, w.wu);
  }
  {
    Scope scope(m, kBDown);
    batch_down_kernel<<<dim3(kH / 16, kDownSplit), kBlock, 0, s>>>(b, w.wd, next_gain);
  }
  return hipGetLastError();
}

hipError_t launch_batch_tail(hipStream_t s, const BatchLaunch &b, const BatchTail &t, Marker *m) {
  if (!batch_shape_ok(b) || t.vocab <= 0) return hipErrorInvalidValue;
  {
    Scope scope(m, kBLmHead);
    batch_lmhead_kernel<<<kBatchLmParts, kLmThreads, 0, s>>>(b, t);
  }
  {
    Scope scope(m, kBArgmax);
    batch_argmax_kernel<<<b.rows, kBlock, 0, s>>>(b, t);
  }
  return hipGetLastError();
}

}  // namespace qd
