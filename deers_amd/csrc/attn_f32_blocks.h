// Blocks of 32 rows of f32 attention operands in LDS and the products of a wave on them, gfx950: what
// attn_split_f32.hip and attn_bwd_f32.hip share.
//
// A wave has LDS for one block of each of its two streamed operands, filled without registers
// (global_load_lds) and read as
//   row fragment     lane l: row l % 32, columns 8 c + 4 g .. + 3 (16-byte reads)
//   column fragment  lane l: column l % 32 of the row in which an accumulator register holds it
// It asks for the next block of an operand as soon as its last product has read the current one.
#pragma once
#include <algorithm>

#include "common.h"

namespace deers {

template <int D>
struct Split32 {
  static constexpr int KH = D / 2;         // elements of D a lane contracts over
  static constexpr int DB = D / 32;        // 32-wide blocks of D
  static constexpr int RB = 4 * D;         // bytes per row
  static constexpr int CH = D / 4;         // 16-byte chunks per row
  static constexpr int NI = CH / 2;        // loads of 1 KB per block
  static constexpr int GP = 1024 + (D == 64 ? 32 : 16);  // LDS pitch of loads
  static constexpr int BB = NI * GP;       // LDS bytes of a 32-row block
  // which row of the block lane group lane / CH of load i has: i * kLoadStep + lane / CH * kLaneStep
  static constexpr int kLoadStep = D == 32 ? 8 : 1, kLaneStep = D == 32 ? 1 : NI;
  static constexpr int at(int row) { return D == 32 ? row / 8 * GP + row % 8 * RB : row % NI * GP + row / NI * RB; }
  static constexpr int kWavesPerSimd = D == 32 ? 3 : D == 64 ? 2 : 1;
};

// A block in LDS is its loads one after the other, 16 or 32 bytes apart, row-major inside a load.  Every
// address is a lane part plus a constant that fits the instruction's offset.  That matters more than
// banks: on this device a vector instruction costs its time beside an f32 matrix instruction, in the
// same wave or another (a backward stage whose addresses were an XOR swizzle took 12.5 K clocks of SIMD
// time for 10.2 K of products).  At head widths 64 and 128 load i has rows i, i + NI, ..., so that of the
// rows which a quarter of a wave reads together at most two share banks; at 32 it has eight rows in
// sequence, four of which do: what a load fetches is then 1 KB in sequence (96 x 1024 x 32 backward 166 us
// against 171).

// Requests rows r0 .. r0 + 31 (rows past T - 1 read row T - 1) of a [T, D] matrix into the block at
// LDS address `dst`.
template <int D>
__device__ __forceinline__ void load_block(const float* base, int row_stride, int r0, int T, uint32_t dst, int lane) {
  using C = Split32<D>;
  const float* row = base + (int64_t)r0 * row_stride;
  const int lane_row = lane / C::CH * C::kLaneStep;
  const uint32_t col_off = 16 * (lane % C::CH);
  if (r0 + 32 <= T) {  // the row of a load goes into its scalar base
    // (opaque: multiples of the step kept for the next call are scalar registers spilled to lanes)
    int step = C::kLoadStep * row_stride;
    asm volatile("" : "+s"(step));
    const uint32_t off = (uint32_t)lane_row * (uint32_t)row_stride * 4 + col_off;
#pragma unroll
    for (int i = 0; i < C::NI; ++i, row += step) async_load16_to_lds(row, off, dst, i * C::GP);
  } else {
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
      async_load16_to_lds(row, (uint32_t)min(i * C::kLoadStep + lane_row, T - 1 - r0) * (uint32_t)row_stride * 4 + col_off,
                          dst, i * C::GP);
  }
}

// This lane's elements of row `row` of a [T, D] matrix in global memory: f[4 c + e] is column
// 8 c + 4 g + e.
template <int D>
__device__ __forceinline__ void row_frag(float (&f)[D / 2], const float* base, int64_t stride, int row, int g) {
  const float* p = base + row * stride + 4 * g;
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    const floatx4 t = *(const floatx4*)(p + 8 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * c + e] = t[e];
  }
}
// c[i][j] += (row i of the block) . (row of lane j, `b`).  With DOT also this lane's share of
// (row lane % 32 of the block) . `other`, its elements in the order of row_frag, from the same reads.
template <int D, bool DOT = false>
__device__ __forceinline__ floatx16 product(uint32_t block, const float (&b)[D / 2], floatx16 c, int lane,
                                            const float* other = nullptr, float* dot = nullptr) {
  using C = Split32<D>;
  const int r = lane & 31;
  const uint32_t at = block + C::at(r) + (lane >> 5) * 16;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < D / 8; ++k) {
    const floatx4 a = lds_read_float4_at(at + 32 * k);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      c = mfma_f32(a[e], b[4 * k + e], c);
      if constexpr (DOT) sum[e] = fmaf(a[e], other[4 * k + e], sum[e]);
    }
  }
  // two reads ahead of the products (left alone, the compiler reads right before each four)
  __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
  for (int k = 0; k < D / 8; ++k) {
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    if (k + 2 < D / 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  if constexpr (DOT) *dot = (sum[0] + sum[1]) + (sum[2] + sum[3]);
  return c;
}
// acc[db] += (columns 32 db .. of the block)^T x: the accumulator `x` as it is is the other operand,
// its register r being row 8 (r / 4) + 4 g + r % 4 of the block.
template <int D>
__device__ __forceinline__ void accumulate(floatx16 (&acc)[D / 32], uint32_t block, const floatx16& x, int lane) {
  using C = Split32<D>;
  const uint32_t at = block + (lane >> 5) * C::at(4) + (lane & 31) * 4;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = 8 * (r >> 2) + (r & 3);
#pragma unroll
    for (int db = 0; db < C::DB; ++db) {
      const float a = *(DEERS_LDS const float*)(uintptr_t)(at + C::at(row) + 128 * db);
      acc[db] = mfma_f32(a, x[r], acc[db]);
    }
  }
  __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
  for (int i = 0; i < 8 * C::DB; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
}

// N results of [32 rows, D] (row = lane % 32) meet by four columns, four registers: every wave leaves its accumulators
// in its own LDS, `own_lds` and on (N * D / 8 KB, no more than its blocks took), and after one barrier wave w adds
// columns w, w + W, .. of all results in wave order, each times its wave's weight where there are any, multiplies by
// mul[n] and writes rows at dst[n] (this lane's row; not where !store).  first_lds: wave 0's, the others' WAVE_BYTES apart.
// 16 bytes per lane both ways; two barriers per result and four bytes took 0.3 us more at D = 32.
template <int D, int W, int N, int WAVE_BYTES>
__device__ __forceinline__ void leave_sums(const floatx16 (&acc)[N][D / 32], uint32_t own_lds, int lane) {
  static_assert(WAVE_BYTES >= N * D * 128, "a wave's sums take its blocks' place");
  if constexpr (W > 1) {
#pragma unroll
    for (int u = 0; u < N * D / 8; ++u) {
      const floatx16& a = acc[u / (D / 8)][u % (D / 8) / 4];
      const int r = u % 4 * 4;
      *(DEERS_LDS floatx4*)(uintptr_t)(own_lds + lane * 16 + u * 1024) = floatx4{a[r], a[r + 1], a[r + 2], a[r + 3]};
    }
  }
  __syncthreads();
}
template <int D, int W, int N, int WAVE_BYTES, bool WEIGHTED = false>
__device__ __forceinline__ void store_sums(const floatx16 (&acc)[N][D / 32], uint32_t first_lds, const float* weight,
                                           const float* mul, float* const* dst, bool store, int wave, int lane) {
  constexpr int U = D / 8;
#pragma unroll
  for (int i = 0; i < N * U / W; ++i) {
    const int u = W == 1 ? i : wave + i * W;
    floatx4 s;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      floatx4 t;
      if constexpr (W == 1) {
        const floatx16& a = acc[i / U][i % U / 4];
        const int r = i % 4 * 4;
        t = floatx4{a[r], a[r + 1], a[r + 2], a[r + 3]};
      } else {
        t = lds_read_float4_at(first_lds + w * WAVE_BYTES + u * 1024 + lane * 16);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = WEIGHTED ? t[e] * weight[w] : t[e];
        s[e] = w ? s[e] + x : x;
      }
    }
    const bool second = N > 1 && u >= U;
    s *= second ? mul[N - 1] : mul[0];
    float* const row = second ? dst[N - 1] : dst[0];
    if (store) *(floatx4*)(row + 32 * (u % U / 4) + 8 * (u % 4) + 4 * (lane >> 5)) = s;
  }
}

template <int D, int W>
constexpr size_t split32_lds() {  // a block of each of two operands per wave, or its sums; row statistics
  return (size_t)W * 2 * Split32<D>::BB + W * 64 * sizeof(float);
}
template <int D, int W>
__device__ __forceinline__ float* split32_stats(char* smem) {
  return (float*)(smem + split32_lds<D, W>() - W * 64 * sizeof(float));
}

// Row statistics from where the lanes have put them, one per row, to the rows of an accumulator.
__device__ __forceinline__ floatx16 stat_rows(const float* stat, int g) {
  floatx16 v;
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    const floatx4 a = *(const floatx4*)(stat + 8 * r4 + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * r4 + e] = a[e];
  }
  return v;
}

}  // namespace deers
