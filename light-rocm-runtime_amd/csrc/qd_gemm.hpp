// FP32 GEMM C = A . W^T on the BF16 matrix cores of gfx950 (device code).
//
// An FP32 number is exactly the sum of three BF16 numbers (8 + 8 + 8
// significant bits): x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0),
// x2 = x - x0 - x1 (exponents below the BF16 range aside, under 2^-102).
// A product a . w is then nine BF16 products; the three smallest (a1 w2,
// a2 w1, a2 w2: below 2^-24 of the product, the rounding of one FP32
// multiplication) are left out and the other six are accumulated in FP32 by
// v_mfma_f32_32x32x16_bf16, which multiplies 16 times as fast as the FP32
// matrix instruction: 2.7 times the FP32 rate after the factor six. The
// leading products a0 w0 have accumulators of their own and the five small ones
// share another, so the sum over k is rounded once per 16 k's instead of once
// per product. BF16 weights are their own first part (three products, exact)
// and FP16 weights two parts (five products).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "qd_device.hpp"
#include "qd_device_math.hpp"

namespace qd {
namespace gemm {

using namespace dev;

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// ---- splitting -----------------------------------------------------------------

// Two floats rounded to BF16 (nearest even), packed low half first.
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2v{x, y}, bf2v));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

// Two floats' three parts, packed (any value: an infinity or one that rounds
// to it leaves NaN in the later parts).
__device__ __forceinline__ void split_pair(float x, float y, uint32_t &h, uint32_t &m, uint32_t &l) {
  h = pack_bf16(x, y);
  const float r0 = x - bf16_lo(h), r1 = y - bf16_hi(h);
  m = pack_bf16(r0, r1);
  l = pack_bf16(r0 - bf16_lo(m), r1 - bf16_hi(m));
}

// Eight floats as three matrix operands.
__device__ __forceinline__ void split_eight(const float (&x)[8], bf8v (&out)[3]) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) split_pair(x[2 * i], x[2 * i + 1], h[i], m[i], l[i]);
  out[0] = __builtin_bit_cast(bf8v, u4v{h[0], h[1], h[2], h[3]});
  out[1] = __builtin_bit_cast(bf8v, u4v{m[0], m[1], m[2], m[3]});
  out[2] = __builtin_bit_cast(bf8v, u4v{l[0], l[1], l[2], l[3]});
}

// The three parts of an operand stored for the GEMM. Unlike the weights'
// split in registers, a value that is not finite keeps itself as its first
// part (the others 0), and one that would round to infinity is truncated, so
// the parts always sum to the value.
struct Parts {
  uint16_t p[3];
};
__device__ __forceinline__ Parts split_value(float x) {
  uint32_t h = pack_bf16(x, 0.f) & 0xFFFFu;
  if ((h & 0x7F80u) == 0x7F80u) h = x != x ? 0x7FC0u : __float_as_uint(x) >> 16;
  const float r = __builtin_isfinite(x) ? x - __uint_as_float(h << 16) : 0.f;
  const uint32_t m = pack_bf16(r, 0.f) & 0xFFFFu;
  const uint32_t l = pack_bf16(r - __uint_as_float(m << 16), 0.f) & 0xFFFFu;
  return {{static_cast<uint16_t>(h), static_cast<uint16_t>(m), static_cast<uint16_t>(l)}};
}
// The value of parts stored by split_value.
__device__ __forceinline__ float join_value(uint16_t h, uint16_t m, uint16_t l) {
  return __uint_as_float(uint32_t(h) << 16) + (__uint_as_float(uint32_t(m) << 16) + __uint_as_float(uint32_t(l) << 16));
}

// The weight operand of one 16-wide k step, this lane's eight consecutive k's
// read from LDS and split into kParts BF16 operands. LDS rows hold kSliceK
// weights in 16-byte slots, slot p of row r holding the row's 16-byte piece
// p ^ swizzle(r), so that the rows of sixteen consecutive lanes at one piece
// fall on distinct banks (256 bytes a clock).
constexpr int kSliceK = 32;  // k's of one LDS stage per k wave
template <typename W>
struct WeightOp;
template <>
struct WeightOp<float> {
  static constexpr int kParts = 3, kSlots = 8;  // 16-byte slots of an LDS row
  __device__ static int swizzle(int row) { return (row >> 1) & 7; }
  __device__ static float widen(const float *p) { return *p; }
  __device__ static void operand(const u4v *row, int sw, int octet, bf8v (&out)[3]) {
    const f4v a = __builtin_bit_cast(f4v, row[(2 * octet) ^ sw]), b = __builtin_bit_cast(f4v, row[(2 * octet + 1) ^ sw]);
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    split_eight(x, out);
  }
};
__device__ __forceinline__ int narrow_swizzle(int row) { return (row >> 2) & 3; }
template <>
struct WeightOp<Bf16> {
  static constexpr int kParts = 1, kSlots = 4;
  __device__ static int swizzle(int row) { return narrow_swizzle(row); }
  __device__ static float widen(const Bf16 *p) { return __uint_as_float(uint32_t(p->bits) << 16); }
  __device__ static void operand(const u4v *row, int sw, int octet, bf8v (&out)[1]) {
    out[0] = __builtin_bit_cast(bf8v, row[octet ^ sw]);
  }
};
template <>
struct WeightOp<F16> {
  static constexpr int kParts = 2, kSlots = 4;
  __device__ static int swizzle(int row) { return narrow_swizzle(row); }
  __device__ static float widen(const F16 *p) { return half_lo(p->bits); }
  __device__ static void operand(const u4v *row, int sw, int octet, bf8v (&out)[2]) {
    const u4v r = row[octet ^ sw];
    u4v h, m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = half_lo(r[i]), y = half_hi(r[i]);
      h[i] = pack_bf16(x, y);
      m[i] = pack_bf16(x - bf16_lo(h[i]), y - bf16_hi(h[i]));
    }
    out[0] = __builtin_bit_cast(bf8v, h);
    out[1] = __builtin_bit_cast(bf8v, m);
  }
};

// ---- the kernel ------------------------------------------------------------------

// A [m][k] as three planes of BF16 parts (row stride lda elements, plane
// stride a_plane); W [n][k] (row stride k). Plain: split z of `splits` over k
// writes its partial product to c + z * m * n. SwiGLU: act = silu(A . w^T) *
// (A . w2^T), n = rows of w, as parts to y (row stride n, plane stride
// y_plane).
template <typename W>
struct Args {
  const uint16_t *a;
  size_t a_plane;
  int lda;
  const W *w, *w2;
  int k, m, n;
  float *c;
  int splits;
  uint16_t *y;
  size_t y_plane;
};

constexpr int kThreads = 256;
constexpr int kStages = 2;  // LDS stages: one is filled while the other is multiplied
constexpr int kDealXcds = 8;  // consecutive workgroups go to consecutive XCDs

typedef __attribute__((address_space(3))) void gemm_lds_void;

// One 16-byte global -> LDS DMA per lane (lane l's bytes land at LDS address
// lds + 16 l). Issued from inline assembly: the compiler would otherwise guard
// every later LDS read with a wait for all DMAs in flight.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is reserved: set before each use, never saved
__device__ __forceinline__ void dma16(const void *src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop
// Workgroup barrier over LDS only: this wave's LDS operations are complete.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Exchanges rows 1 and 3 (of 16 lanes) of a with rows 0 and 2 of b. (The s_nop
// gives the two wait states the swap needs after a VALU write.)
__device__ __forceinline__ void row_swap(float &a, float &b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}

// Output element (row, col) over k's [k0, k1) in FP32: where the split
// product is not finite (an operand was not, or an overflow), the element is
// what FP32 arithmetic gives.
template <typename W>
__device__ __forceinline__ float fp32_element(const Args<W> &g, int row, const W *wrow, int k0, int k1) {
  const uint16_t *a = g.a + static_cast<size_t>(row) * g.lda;
  float s = 0.f;
  for (int k = k0; k < k1 && s == s; ++k)
    s = fmaf(join_value(a[k], a[g.a_plane + k], a[2 * g.a_plane + k]), WeightOp<W>::widen(wrow + k), s);
  return s;
}

// Waits for this wave's DMAs.
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Workgroup of four waves, WM along m, WN along n and WK along k; a wave
// multiplies RB blocks of 32 x 32, so the output tile is 32 RB WM rows by 32 WN
// columns (SwiGLU: 16 WN gate columns and the same up columns). A's parts and
// W's values go through the LDS stages, 32 WK k's each, by DMA; a wave splits the
// weights it reads. WK waves' partial tiles are summed through LDS in k order.
// Operand layout of v_mfma_f32_32x32x16_bf16: lane l supplies A[l % 32] and
// B[l % 32] at k's 8 (l / 32) .. + 7; accumulator register r of lane l holds
// D[(r / 4) * 8 + (l / 32) * 4 + r % 4][l % 32].
template <int RB, int WM, int WN, int WK, typename W, bool kSwiGLU>
__global__ __launch_bounds__(kThreads, 2) void gemm_split_kernel(Args<W> g, int mtiles, int pairs) {
  static_assert(WM * WN * WK == 4, "four waves");
  using Op = WeightOp<W>;
  constexpr int kRows = 32 * RB * WM, kCols = 32 * WN;
  constexpr int kPlane = kRows * kSliceK * 2;               // bytes of one plane of one k wave's slice
  constexpr int kWRow = kSliceK * static_cast<int>(sizeof(W));  // bytes of a weight row's slice
  constexpr int kABytes = WK * 3 * kPlane, kStage = kABytes + WK * kCols * kWRow;
  constexpr int kReduce = WK > 1 ? 4 * RB * 16 * kWave * 4 : 0;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kStages * kStage > kReduce ? kStages * kStage : kReduce];

  // Workgroups of one (column tile, split) pair, which read the same weights,
  // are dealt to one XCD, next to each other in its order.
  const int x = blockIdx.x % kDealXcds, q = blockIdx.x / kDealXcds;
  const int pair = (q / mtiles) * kDealXcds + x, m0 = (q % mtiles) * kRows;
  if (pair >= pairs) return;
  const int tile = pair / g.splits, z = pair % g.splits;
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
  const int wn = w % WN, wm = (w / WN) % WM, wk = w / (WN * WM);
  const int half = lane >> 5, lr = lane & 31;
  const int slices = g.k / (kSliceK * WK);
  const int s0 = z * slices / g.splits, n = (z + 1) * slices / g.splits - s0;

  // Weight row of the tile's column c (SwiGLU: 16 gate rows, then the 16 up
  // rows of the same activations, in each block of 32).
  auto weight_row = [&](int c) {
    if constexpr (kSwiGLU)
      return ((c & 31) < 16 ? g.w : g.w2) + static_cast<size_t>((tile * (kCols / 32) + c / 32) * 16 + (c & 15)) * g.k;
    else
      return g.w + static_cast<size_t>(tile * kCols + c) * g.k;
  };
  // The stage's DMAs of 1 KiB, dealt to the waves in turn: A's in pieces of 16
  // rows of one plane, then W's in pieces of 8 (FP32) or 16 rows. (A wave
  // without one of the last repeats the last: the same bytes to the same place.)
  constexpr int kAGroups = kABytes / 1024, kGroups = kStage / 1024, kIssue = (kGroups + 3) / 4;
  constexpr int kWGroupRows = 64 / Op::kSlots, kWGroupsK = kCols / kWGroupRows;
  const uint32_t lds_base = static_cast<uint32_t>(
      __builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>((gemm_lds_void *)lds))));
  const unsigned char *src[kIssue];
#pragma unroll
  for (int i = 0; i < kIssue; ++i) {
    const int gi = min(w + 4 * i, kGroups - 1);
    if (gi < kAGroups) {
      const int pk = gi / (kRows / 16), rg = gi % (kRows / 16);  // pk = k wave * 3 + plane
      const int row = 16 * rg + (lane >> 2);
      const int oct = (lane & 3) ^ narrow_swizzle(row);
      src[i] = reinterpret_cast<const unsigned char *>(
          g.a + static_cast<size_t>(pk % 3) * g.a_plane + static_cast<size_t>(min(m0 + row, g.m - 1)) * g.lda +
          (s0 * WK + pk / 3) * kSliceK + 8 * oct);
    } else {
      const int kk = (gi - kAGroups) / kWGroupsK, rg = (gi - kAGroups) % kWGroupsK;
      const int row = kWGroupRows * rg + lane / Op::kSlots;
      const int piece = (lane % Op::kSlots) ^ Op::swizzle(row);
      src[i] = reinterpret_cast<const unsigned char *>(weight_row(row) + (s0 * WK + kk) * kSliceK) + 16 * piece;
    }
  }
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < kIssue; ++i) {
      const int gi = min(w + 4 * i, kGroups - 1);
      dma16(src[i], lds_base + b * kStage + gi * 1024);
      src[i] += gi < kAGroups ? WK * kSliceK * 2 : WK * kWRow;
    }
  };

  // Sums of many leading products are rounded at their own size, so they are
  // kept short: where a wave multiplies all of its split's k's, their chain
  // (lead[0]) is added to a total (lead[1]) every kFold slices; else, at most 14
  // slices to a wave, two chains take every other 16 k's each.
  // Errors of the last of two layers' K rows against 64 bits, two chains (beyond
  // 1,024 rows one) / folded / a step per token, 1e-7, BF16: 200 rows 3.22 / 2.92
  // / 3.11, 512 3.44 / 3.18 / 3.18, 1,000 3.92 / 3.64 / 3.58; the logits of 1,999
  // rows 12.6 / 8.5 / 7.1. It costs 0.5 % of a 512-row prompt, 1.5 % of 200 rows
  // in F16 and 1.6 % of 1,999 rows (folding every 4 slices there: 2.2 %, 8.4).
  // The 128-row tile has registers for the total only if it holds the operands
  // of kAtOnce blocks of rows at a time (all four: 30 spilt, 13.9 ms for 1,999
  // rows instead of 11.3).
  constexpr bool kFolds = WK == 1;
  constexpr int kFold = RB < 4 ? 4 : 8, kAtOnce = RB < 4 ? RB : 1;
  f16v lead[2][RB] = {}, tail[RB] = {};
  if (n > 0) fetch(0);
  int b = 0, s = 0;
  auto slice = [&] {
    // This wave's part of slice s has landed; after the barrier every wave's
    // has, and every wave is done with the slice before, whose stage is filled
    // next. (With the stages as b and b ^ 1 the F16 kernels are 1 % slower.)
    dma_wait();
    lds_barrier();
    if (s + 1 < n) fetch(b == 0 ? kStages - 1 : b - 1);
    const unsigned char *st = lds + b * kStage;
    b = b + 1 == kStages ? 0 : b + 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf8v wv[Op::kParts];
      const int c = 32 * wn + lr;
      Op::operand(reinterpret_cast<const u4v *>(st + kABytes + (wk * kCols + c) * kWRow), Op::swizzle(c), 2 * j + half,
                  wv);
#pragma unroll
      for (int r0 = 0; r0 < RB; r0 += kAtOnce) {
        bf8v av[kAtOnce][3];
#pragma unroll
        for (int r = 0; r < kAtOnce; ++r) {
          const int row = 32 * (wm * RB + r0 + r) + lr;
          const int slot = (2 * j + half) ^ narrow_swizzle(row);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            av[r][p] = *reinterpret_cast<const bf8v *>(st + (wk * 3 + p) * kPlane + row * kSliceK * 2 + 16 * slot);
        }
        auto mac = [&](f16v (&acc)[RB], int pa, int pw) {
#pragma unroll
          for (int r = 0; r < kAtOnce; ++r)
            acc[r0 + r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[r][pa], wv[pw], acc[r0 + r], 0, 0, 0);
        };
        mac(lead[kFolds ? 0 : j], 0, 0);
        if constexpr (Op::kParts > 1) mac(tail, 0, 1);
        mac(tail, 1, 0);
        if constexpr (Op::kParts > 1) mac(tail, 1, 1);
        if constexpr (Op::kParts > 2) mac(tail, 0, 2);
        mac(tail, 2, 0);
      }
    }
  };
  while (s < n) {
    const int end = kFolds ? min(n, s + kFold) : n;
    for (; s < end; ++s) slice();
    if constexpr (kFolds) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        lead[1][rb] += lead[0][rb];
        lead[0][rb] = f16v{};
      }
    }
  }

  // The wave's elements of the tile: all, or with WK waves along k the 1 / WK
  // of the accumulator registers that this wave finishes.
  constexpr int kRegs = RB * 16 / WK;
  float v[kRegs];
  auto sum = [&](int i) {
    return (lead[0][i / 16][i % 16] + lead[1][i / 16][i % 16]) + tail[i / 16][i % 16];
  };
  if constexpr (WK == 1) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) v[i] = sum(i);
  } else {
    float *red = reinterpret_cast<float *>(lds);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RB * 16; ++i) red[(w * RB * 16 + i) * kWave + lane] = sum(i);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      v[i] = 0.f;
#pragma unroll
      for (int u = 0; u < WK; ++u)
        v[i] += red[((u * WM * WN + wm * WN + wn) * RB * 16 + wk * kRegs + i) * kWave + lane];
    }
  }
  // Column of the wave's elements and row of element i within the tile.
  const int tile_col = 32 * wn + lr;
  auto tile_row = [&](int i) {
    const int r = wk * kRegs + i;
    return 32 * (wm * RB + r / 16) + ((r % 16) / 4) * 8 + half * 4 + r % 4;
  };
  float probe = 0.f;  // 0 as long as every element is finite
#pragma unroll
  for (int i = 0; i < kRegs; ++i) probe = fmaf(v[i], 0.f, probe);
  if (probe != 0.f) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i)
      if (!__builtin_isfinite(v[i]) && m0 + tile_row(i) < g.m)
        v[i] = fp32_element(g, m0 + tile_row(i), weight_row(tile_col), s0 * WK * kSliceK, (s0 + n) * WK * kSliceK);
  }
  if constexpr (kSwiGLU) {
    // Elements i and i + 1 are adjacent rows; lanes lr < 16 hold their gate
    // sums and lanes lr + 16 the up sums of the same activations. One swap
    // gives the former both sums of row i and the latter both of row i + 1.
#pragma unroll
    for (int i = 0; i < kRegs; i += 2) {
      row_swap(v[i], v[i + 1]);
      const int row = m0 + tile_row(i) + (lr >> 4);
      const Parts out = split_value(silu_mul(v[i], v[i + 1]));
      if (row < g.m) {
        uint16_t *y = g.y + static_cast<size_t>(row) * g.n + (tile * (kCols / 32) + wn) * 16 + (lr & 15);
        y[0] = out.p[0];
        y[g.y_plane] = out.p[1];
        y[2 * g.y_plane] = out.p[2];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      const int row = m0 + tile_row(i);
      if (row < g.m) g.c[(static_cast<size_t>(z) * g.m + row) * g.n + tile * kCols + tile_col] = v[i];
    }
  }
}

}  // namespace gemm
}  // namespace qd
