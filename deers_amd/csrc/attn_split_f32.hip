// Fused causal attention of up to middling launches, f32 storage and arithmetic, gfx950: forward and
// backward of the same contract as attn_fwd_f32.hip and attn_bwd_f32.hip
// (src/models/gpt.rs:139-144; src/ops.rs:1089-1101, 422-425, 210-214, 777-799, 1162-1175, 638-643).
//
// The kernels of those files give a workgroup 128 rows whose four waves walk the other operand
// together, a chain of T / 32 stages with barriers, and the backward is two or three launches.  Here
// a workgroup owns 32 rows and its W waves divide the 32-row blocks of the other operand (wave w
// takes blocks w, w + W, ...), without a barrier until their partial sums meet at the end, so the
// chain of a wave is T / (32 W) stages and four times as many workgroups are in flight.
//
//   forward  S^T = K Q^T, O^T += V^T P^T; online softmax per wave; O, m and l are merged.
//   dQ       dP^T = V dO^T, S^T, dQ^T += K^T dS^T; sums merged.
//   dK/dV    a workgroup owns 32 keys: dP = dO V^T, S = Q K^T, dV^T += dO^T P, dK^T += Q^T dS.  It forms
//            each query block's row sums dO . O itself: no workspace, no hand-over.
// The backward computes S and dP twice, 7 products per block against the one-pass kernel's 5: the
// price of one launch whose workgroups wait for nobody.  Partial sums are added in wave order:
// dQ, dK and dV are reproducible bit for bit.
//
// A wave's first loads and its merge cost it some 10 K clocks; blocks are dealt so that every XCD has
// the same number of them also when the heads are not a multiple of eight (map_block_even).
//
// A product costs 64 clocks of matrix pipe per two elements of D (v_mfma_f32_32x32x2_f32), so the
// pipe is the bound as long as a wave's blocks arrive in time.  Each wave has LDS for one block of
// each of its two streamed operands, filled without registers (global_load_lds) and read as
//   row fragment     lane l: row l % 32, columns 8 c + 4 g .. + 3 (16-byte reads)
//   column fragment  lane l: column l % 32 of the row in which an accumulator register holds it
// and asks for the next block of an operand as soon as its last product has read the current one:
// the operand whose block is asked for last is the one that the next stage needs second, so that
// both requests are covered by a product (2048 clocks at D = 64).  A lone wave's dK/dV stage takes
// 12.3 K clocks for 8.2 K of products (D = 64); two waves per SIMD run at 84 % of the pipe.
//
// us, forward / backward, 128-row kernels -> these: 24 heads x 256 x 32 15.4 / 26.1 -> 6.1 / 12.2, 12 x 512 x 64
// 41 / 66 -> 14 / 33, 12 x 1024 x 64 77 / 121 -> 29 / 70, 3 x 4096 x 32 191 / 337 -> 55 / 131, 15 x 777 x 128 120 / 403
// -> 40 / 140, 800 x 128 x 64 49 / 134 -> 35 / 99.
#include <algorithm>

#include "common.h"

namespace deers {

namespace {

#define ZERO16S floatx16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}

template <int D>
struct Split32 {
  static constexpr int KH = D / 2;         // elements of D a lane contracts over
  static constexpr int DB = D / 32;        // 32-wide blocks of D
  static constexpr int RB = 4 * D;         // bytes per row
  static constexpr int CH = D / 4;         // 16-byte chunks per row
  static constexpr int BB = 32 * RB;       // bytes of a 32-row block
  static constexpr int NI = BB / 1024;     // loads per block
  static constexpr int kWavesPerSimd = D == 32 ? 3 : D == 64 ? 2 : 1;
};

// Chunk c of row r of a block sits at position c ^ swizzle(r): 16 consecutive rows read at one chunk
// hit 16 different 16-byte bank groups, and two rows 4 apart read along their columns different halves.
// Linear over XOR, so an address is a lane part, computed once per use of a block, XOR a constant
// (blocks are aligned to their size).  The lane parts are kept from the optimiser, which would
// otherwise compute some eighty addresses before the loop and spill them.
template <int D>
__device__ __forceinline__ int swizzle32(int r) {
  if constexpr (D == 32) return (r >> 1) & 7;
  return (r & 3) | ((r >> 1) & 4) | ((r << 1) & 8);
}

// Before the loads into a block that earlier LDS reads of this wave have used: those have returned.
__device__ __forceinline__ void settle_lds_reads() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
}

// Requests rows r0 .. r0 + 31 (rows past T - 1 read row T - 1) of a [T, D] matrix into the block at
// LDS address `dst`.
template <int D>
__device__ __forceinline__ void load_block(const float* base, int row_stride, int r0, int T, uint32_t dst, int lane) {
  using C = Split32<D>;
  const int lane_row = lane / C::CH, lane_chunk = (lane % C::CH) ^ swizzle32<D>(lane_row);
  constexpr int RPL = 64 / C::CH;  // rows per load
  if (r0 + 32 <= T) {  // the row of a load goes into its scalar base
    const uint32_t row_off = opaque((uint32_t)lane_row * (uint32_t)row_stride * 4);
    const float* row = base + (int64_t)r0 * row_stride;
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
      async_load16_to_lds(row + (int64_t)(i * RPL) * row_stride,
                          row_off + 16 * (lane_chunk ^ swizzle32<D>(i * RPL)), dst + i * 1024);
  } else {
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
      async_load16_to_lds(base, (uint32_t)min(r0 + i * RPL + lane_row, T - 1) * (uint32_t)row_stride * 4 +
                                    16 * (lane_chunk ^ swizzle32<D>(i * RPL)), dst + i * 1024);
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
// (row lane % 32 of the block) . `other`, its elements in the order of row_frag: vector work that runs
// under the products.
template <int D, bool DOT = false>
__device__ __forceinline__ floatx16 product(uint32_t block, const float (&b)[D / 2], floatx16 c, int lane,
                                            const float* other = nullptr, float* dot = nullptr) {
  using C = Split32<D>;
  const int r = lane & 31;
  const uint32_t at = opaque(block + r * C::RB + (((lane >> 5) ^ swizzle32<D>(r)) << 4));
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < D / 8; ++k) {
    const floatx4 a = lds_read_float4_at(at ^ (32 * k));
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
  const int g = lane >> 5;
  const uint32_t at = opaque(block + 4 * g * C::RB + ((swizzle32<D>(4 * g) << 4) ^ ((lane & 31) * 4)));
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = 8 * (r >> 2) + (r & 3);
#pragma unroll
    for (int db = 0; db < C::DB; ++db) {
      const float a = *(DEERS_LDS const float*)(uintptr_t)((at ^ (128 * db) ^ (swizzle32<D>(row) << 4)) + row * C::RB);
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

// Adds the W waves' accumulators of a [32 rows, D] result (row = lane % 32), each scaled by its
// wave's `weight` first, in wave order, multiplies by `mul` and writes rows at dst (this lane's
// row; not where !store).  `red` is LDS for W * D / 2 * 64 floats.  Starts with a barrier.
template <int D, int W>
__device__ __forceinline__ void merge_store(const floatx16 (&acc)[D / 32], float weight, float mul, float* dst,
                                            bool store, float* red, int wave, int lane) {
  __syncthreads();
#pragma unroll
  for (int r = 0; r < D / 2; ++r) red[(wave * (D / 2) + r) * 64 + lane] = acc[r / 16][r % 16] * weight;
  __syncthreads();
#pragma unroll
  for (int u = wave; u < D / 8; u += W) {  // registers 4 u .. 4 u + 3: four columns
    floatx4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float t = red[(4 * u + e) * 64 + lane];
#pragma unroll
      for (int w = 1; w < W; ++w) t += red[(w * (D / 2) + 4 * u + e) * 64 + lane];
      s[e] = t * mul;
    }
    if (store) *(floatx4*)(dst + 32 * (u / 4) + 8 * (u % 4) + 4 * (lane >> 5)) = s;
  }
}

template <int D, int W>
constexpr size_t split32_lds() {  // a block of each of two operands per wave, or the merge; row statistics
  return std::max((size_t)W * 2 * Split32<D>::BB, (size_t)W * (D / 2) * 64 * sizeof(float)) + W * 64 * sizeof(float);
}
template <int D, int W>
__device__ __forceinline__ float* split32_stats(char* smem) {
  return (float*)(smem + split32_lds<D, W>() - W * 64 * sizeof(float));
}

// ---- forward ----

template <int D, int W>
__global__ __launch_bounds__(64 * W, Split32<D>::kWavesPerSimd) void attn_fwd_f32_split_kernel(FwdParams p, int BH, int n_blocks) {
  using C = Split32<D>;
  constexpr int KH = C::KH, DB = C::DB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, T = p.T;
  int bh, rank;
  if (!map_block_even(blockIdx.x, n_blocks, BH, &bh, &rank)) return;
  const int qb = n_blocks - 1 - rank;  // longest rows first
  const int b = bh / p.H, h = bh % p.H;
  const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
  const float* V = (const float*)p.v + b * p.sv.b + h * p.sv.h;
  const int skt = (int)p.sk.t, svt = (int)p.sv.t;
  const int qrow = 32 * qb + (lane & 31);
  const uint32_t k_blk = lds_address(smem) + wave * 2 * C::BB, v_blk = k_blk + C::BB;

  float qf[KH];
  row_frag<D>(qf, (const float*)p.q + b * p.sq.b + h * p.sq.h, p.sq.t, min(qrow, T - 1), g);
  int kb = wave;
  if (kb <= qb) {
    load_block<D>(K, skt, 32 * kb, T, k_blk, lane);
    load_block<D>(V, svt, 32 * kb, T, v_blk, lane);
  }
  wait_all_vmem();
#pragma unroll
  for (int k = 0; k < KH; ++k) qf[k] *= p.scale_log2;

  floatx16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = ZERO16S;
  float m = -INFINITY, l = 0.f;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    wait_vmcnt<C::NI>();  // K; V's block may be on its way
    floatx16 s = product<D>(k_blk, qf, ZERO16S, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(K, skt, 32 * (kb + W), T, k_blk, lane);
    }
    if (kb == qb) {  // the diagonal block (its keys past T - 1 lie in the future of every stored row)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
    float mx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) mx[i] = fmaxf(fmaxf(s[i], s[i + 4]), fmaxf(s[i + 8], s[i + 12]));
    const float m_new = fmaxf(m, pair_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]))));
    const float alpha = fast_exp2(m - m_new);  // 0 in the first block
    m = m_new;
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - m);
      sum[r & 1] += s[r];
    }
    l = l * alpha + (sum[0] + sum[1]);
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
    if (more)
      wait_vmcnt<C::NI>();  // V
    else
      wait_vmcnt<0>();
    accumulate<D>(oacc, v_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(V, svt, 32 * (kb + W), T, v_blk, lane);
    }
  }

  // ---- the waves' (m, l, O) become one; a wave without a block has m = -inf and weight 0 ----
  float* stat_m = split32_stats<D, W>(smem);
  float* stat_l = stat_m + W * 32;
  l = pair_sum(l);
  if (g == 0) {
    stat_m[wave * 32 + lane] = m;
    stat_l[wave * 32 + lane] = l;
  }
  __syncthreads();
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) M = fmaxf(M, stat_m[w * 32 + (lane & 31)]);
#pragma unroll
  for (int w = 0; w < W; ++w) L += stat_l[w * 32 + (lane & 31)] * fast_exp2(stat_m[w * 32 + (lane & 31)] - M);
  float* orow = (float*)p.o + b * p.so.b + h * p.so.h + (int64_t)min(qrow, T - 1) * p.so.t;
  merge_store<D, W>(oacc, fast_exp2(m - M), 1.f / L, orow, qrow < T, (float*)smem, wave, lane);
  if (wave == 0 && g == 0 && qrow < T) p.lse[(int64_t)bh * T + qrow] = (M + fast_log2(L)) * kLn2;
}

// ---- backward ----

template <int D, int W>
__device__ __forceinline__ void split32_dq(const BwdParams& p, int bh, int qb, char* smem, int wave, int lane) {
  using C = Split32<D>;
  constexpr int KH = C::KH, DB = C::DB;
  const int g = lane >> 5, T = p.T;
  const int b = bh / p.H, h = bh % p.H;
  const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
  const float* V = (const float*)p.v + b * p.sv.b + h * p.sv.h;
  const int skt = (int)p.sk.t, svt = (int)p.sv.t;
  const int qrow = 32 * qb + (lane & 31), qread = min(qrow, T - 1);
  const uint32_t k_blk = lds_address(smem) + wave * 2 * C::BB, v_blk = k_blk + C::BB;

  float qf[KH], dof[KH];
  float nd;
  const float lse = p.lse[(int64_t)bh * T + qread];
  int kb = wave;
  {
    float of[KH];
    row_frag<D>(of, (const float*)p.o + b * p.so.b + h * p.so.h, p.so.t, qread, g);
    row_frag<D>(dof, (const float*)p.d_o + b * p.sdo.b + h * p.sdo.h, p.sdo.t, qread, g);
    row_frag<D>(qf, (const float*)p.q + b * p.sq.b + h * p.sq.h, p.sq.t, qread, g);
    if (kb <= qb) {
      load_block<D>(V, svt, 32 * kb, T, v_blk, lane);
      load_block<D>(K, skt, 32 * kb, T, k_blk, lane);
    }
    wait_all_vmem();
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KH; ++k) s[k & 3] = fmaf(of[k], dof[k], s[k & 3]);
    nd = -pair_sum((s[0] + s[1]) + (s[2] + s[3]));
  }
  const float lse2 = -lse * kLog2e;
#pragma unroll
  for (int k = 0; k < KH; ++k) qf[k] *= p.scale_log2;

  floatx16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[db] = ZERO16S;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    floatx16 s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = lse2;
      dp[r] = nd;
    }
    wait_vmcnt<C::NI>();  // V; K's block may be on its way
    dp = product<D>(v_blk, dof, dp, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(V, svt, 32 * (kb + W), T, v_blk, lane);
      wait_vmcnt<C::NI>();  // K
    } else {
      wait_vmcnt<0>();
    }
    s = product<D>(k_blk, qf, s, lane);
    if (kb == qb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r]) * dp[r];
    accumulate<D>(dq, k_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(K, skt, 32 * (kb + W), T, k_blk, lane);
    }
  }
  float* row = (float*)p.dq + b * p.sdq.b + h * p.sdq.h + (int64_t)qread * p.sdq.t;
  merge_store<D, W>(dq, 1.f, p.scale, row, qrow < T, (float*)smem, wave, lane);
}

template <int D, int W>
__device__ __forceinline__ void split32_dkdv(const BwdParams& p, int bh, int kb, int n_blocks, char* smem, int wave,
                                             int lane) {
  using C = Split32<D>;
  constexpr int KH = C::KH, DB = C::DB;
  const int g = lane >> 5, T = p.T;
  const int b = bh / p.H, h = bh % p.H;
  const float* Q = (const float*)p.q + b * p.sq.b + h * p.sq.h;
  const float* O = (const float*)p.o + b * p.so.b + h * p.so.h;
  const float* dO = (const float*)p.d_o + b * p.sdo.b + h * p.sdo.h;
  const float* lse = p.lse + (int64_t)bh * T;
  const int sqt = (int)p.sq.t, sdot = (int)p.sdo.t;
  const int krow = 32 * kb + (lane & 31), kread = min(krow, T - 1);
  const uint32_t q_blk = lds_address(smem) + wave * 2 * C::BB, do_blk = q_blk + C::BB;
  float* stat = split32_stats<D, W>(smem) + wave * 64;

  float kf[KH], vf[KH];
  row_frag<D>(kf, (const float*)p.k + b * p.sk.b + h * p.sk.h, p.sk.t, kread, g);
  row_frag<D>(vf, (const float*)p.v + b * p.sv.b + h * p.sv.h, p.sv.t, kread, g);
  int qb = kb + wave;
  if (qb < n_blocks) {
    load_block<D>(Q, sqt, 32 * qb, T, q_blk, lane);
    load_block<D>(dO, sdot, 32 * qb, T, do_blk, lane);
  }
  wait_all_vmem();
#pragma unroll
  for (int k = 0; k < KH; ++k) kf[k] *= p.scale_log2;

  floatx16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dk[db] = dv[db] = ZERO16S;
  for (; qb < n_blocks; qb += W) {
    const bool more = qb + W < n_blocks;
    const int row = 32 * qb + (lane & 31), read = min(row, T - 1);
    float of[KH], sum;
    row_frag<D>(of, O, p.so.t, read, g);  // used under the second product
    const float lse_row = lse[read];
    wait_vmcnt<2 * C::NI + 1>();  // Q; dO's block may be on its way
    floatx16 s = product<D>(q_blk, kf, ZERO16S, lane);
    wait_vmcnt<C::NI + 1>();  // dO
    floatx16 dp = product<D, true>(do_blk, vf, ZERO16S, lane, of, &sum);
    // the block's row statistics, from the lanes that hold them to the rows of the accumulators
    sum = pair_sum(sum);
    if (g == 0) {
      stat[lane] = row < T ? -lse_row * kLog2e : -INFINITY;  // a padded query's probabilities are zero
      stat[32 + lane] = -sum;
    }
    if (qb == kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) < (lane & 31)) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 l4 = *(const floatx4*)(stat + 8 * r4 + 4 * g), d4 = *(const floatx4*)(stat + 32 + 8 * r4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = fast_exp2(s[4 * r4 + e] + l4[e]);
        s[4 * r4 + e] = pv;
        dp[4 * r4 + e] = pv * (dp[4 * r4 + e] + d4[e]);
      }
    }
    accumulate<D>(dk, q_blk, dp, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(Q, sqt, 32 * (qb + W), T, q_blk, lane);
    }
    accumulate<D>(dv, do_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(dO, sdot, 32 * (qb + W), T, do_blk, lane);
    }
  }
  float* dv_row = (float*)p.dv + b * p.sdv.b + h * p.sdv.h + (int64_t)kread * p.sdv.t;
  float* dk_row = (float*)p.dk + b * p.sdk.b + h * p.sdk.h + (int64_t)kread * p.sdk.t;
  merge_store<D, W>(dv, 1.f, 1.f, dv_row, krow < T, (float*)smem, wave, lane);
  merge_store<D, W>(dk, 1.f, p.scale, dk_row, krow < T, (float*)smem, wave, lane);
}

// Ranks alternate between the roles, longest first: rank 2 r is the dK/dV block of keys 32 r ..,
// rank 2 r + 1 the dQ block as many rows from the end.
template <int D, int W>
__global__ __launch_bounds__(64 * W, Split32<D>::kWavesPerSimd) void attn_bwd_f32_split_kernel(BwdParams p, int BH, int n_blocks) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, rank;
  if (!map_block_even(blockIdx.x, 2 * n_blocks, BH, &bh, &rank)) return;
  if (rank & 1)
    split32_dq<D, W>(p, bh, n_blocks - 1 - (rank >> 1), smem, wave, lane);
  else
    split32_dkdv<D, W>(p, bh, rank >> 1, n_blocks, smem, wave, lane);
}

template <typename Kernel>
void allow_lds(Kernel kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <int D, int W>
void launch_fwd_split(const FwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_fwd_f32_split_kernel<D, W>;
  constexpr size_t lds = split32_lds<D, W>();
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  hipLaunchKernelGGL(kernel, dim3(map_even_blocks(n_blocks, BH)), dim3(64 * W), lds, stream, p, BH, n_blocks);
}
template <int D, int W>
void launch_bwd_split(const BwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_bwd_f32_split_kernel<D, W>;
  constexpr size_t lds = split32_lds<D, W>();
  static bool attr_set = false;
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  hipLaunchKernelGGL(kernel, dim3(map_even_blocks(2 * n_blocks, BH)), dim3(64 * W), lds, stream, p, BH, n_blocks);
}

}  // namespace

// Which launches come here and with how many waves per workgroup.  Measured on T = 32 .. 8192, 3 ..
// 800 heads and the three head widths against the 128-row kernels and between 1, 2 and 4 waves;
// nb = T / 32 is the length of a walk, n = heads * nb the number of workgroups.
//
// Waves.  Few workgroups: four waves, the shortest chain (D = 64, 12 x 512: forward 14 us, with two
// waves 23, with one 41).  Many: the SIMDs are covered anyway, and a wave that walks longer pays
// its start-up and its merge less often (32 x 12 x 256 x 64: 61 / 51 / 50 us in 4 / 2 / 1).  Never
// more waves than blocks to walk.
//
// Takes, forward: at head width 32, and for walks of up to eight blocks, always.  Otherwise up to
// the size where the 128-row kernel's four-fold reuse of a K/V tile decides: every wave here
// fetches its own blocks (D = 64: 4 x 12 x 1024 69 us against 80, 8 x 12 x 1024 129 against 129, 16 x 12 x
// 768 158 against 150).
// Takes, backward: two more products per block than the one-pass kernel against a launch less,
// no barriers and no atomics: up to about 74 K blocks (D = 64: 12 x 512 33 us against 66, 6 x 12 x 1024
// 303 against 316, 8 x 12 x 1024 380 against 367), or few enough workgroups that the other leaves CUs
// idle (11 x 3000 385 against 477); at head width 32 the products weigh less (8 x 12 x 2048 714
// against 724).
bool attn_fwd_f32_split_takes(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (D == 32 || nb <= 8) return true;
  return D == 128 ? n <= 1536 : n <= 2048 || (nb >= 64 && n <= 3072);
}
bool attn_bwd_f32_split_takes(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (D == 32) return n <= 8192 && n * nb <= 400000;
  return n * nb <= 74000 || n * D / 64 <= 1100;
}
static int fwd_waves(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (n <= 512) return nb >= 4 ? 4 : nb >= 2 ? 2 : 1;
  if (nb >= 12 && D <= 64) return n <= 8192 ? 4 : 1;
  return n <= 1536 && nb >= 4 ? 2 : 1;
}
static int bwd_waves(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb, u = n * D / 64;
  const int64_t most = u > 320 ? nb / 2 : nb;
  const int64_t w = u <= 640 || (u <= 1100 && nb >= 32) ? 4 : u <= 1536 ? 2 : 1;
  return (int)(std::min(w, most) >= 4 ? 4 : std::min(w, most) >= 2 ? 2 : 1);
}

template <int W>
static void launch_fwd(const FwdParams& p, int BH, int D, hipStream_t stream) {
  switch (D) {
    case 32: launch_fwd_split<32, W>(p, BH, stream); break;
    case 64: launch_fwd_split<64, W>(p, BH, stream); break;
    case 128: launch_fwd_split<128, W>(p, BH, stream); break;
  }
}
template <int W>
static void launch_bwd(const BwdParams& p, int BH, int D, hipStream_t stream) {
  switch (D) {
    case 32: launch_bwd_split<32, W>(p, BH, stream); break;
    case 64: launch_bwd_split<64, W>(p, BH, stream); break;
    case 128: launch_bwd_split<128, W>(p, BH, stream); break;
  }
}

void launch_attn_fwd_f32_split(const FwdParams& p, int B, int D, hipStream_t stream) {
  LaunchScope scope("attn_fwd_f32", stream);
  switch (fwd_waves((int64_t)B * p.H, p.T, D)) {
    case 1: launch_fwd<1>(p, B * p.H, D, stream); break;
    case 2: launch_fwd<2>(p, B * p.H, D, stream); break;
    case 4: launch_fwd<4>(p, B * p.H, D, stream); break;
  }
}
void launch_attn_bwd_f32_split(const BwdParams& p, int B, int D, hipStream_t stream) {
  LaunchScope scope("attn_bwd_f32", stream);
  switch (bwd_waves((int64_t)B * p.H, p.T, D)) {
    case 1: launch_bwd<1>(p, B * p.H, D, stream); break;
    case 2: launch_bwd<2>(p, B * p.H, D, stream); break;
    case 4: launch_bwd<4>(p, B * p.H, D, stream); break;
  }
}

}  // namespace deers
