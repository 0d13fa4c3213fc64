// Fused causal attention for launches that cannot fill the device, f16 storage / f32
// accumulate, gfx950: forward and backward of the same contract as attn_fwd_f16.hip and
// attn_bwd_f16.hip (src/models/gpt.rs:139-144; src/ops.rs:1089-1101, 422-425, 210-214, 777-799,
// 1162-1175, 638-643).
//
// The kernels of those files give a workgroup 128 rows and let its four waves walk the other
// operand together: one dependent chain of T / 32 stages with a barrier in each.  With few heads
// or short sequences the launch is nothing but that chain (12 heads of 512 x 64: 48 workgroups on
// 256 CUs, forward 10.1 us and backward 17.5 us; here 6.4 and 10.9).  Here a workgroup owns 32 rows,
// so there are four times as many of them, and its W waves divide the blocks of 32 rows of the
// other operand among themselves (wave w takes blocks w, w + W, ...), each with its own loads,
// its own slice of LDS and no barrier; their partial results meet once, at the end, in LDS.  The
// chain of a wave is T / (32 W) stages.  The price is that nothing is shared between waves: every
// 32 rows read all of the other operand through L1 (64 bytes per clock and CU), so launches that
// fill the device anyway stay with the 128-row kernels (the rule is above split_takes, below).
//
//   forward  S^T = K Q^T, one query per lane; V through LDS for its transposed fragments, K through
//            LDS or straight into registers; online softmax per wave; O, m and l are merged.
//   dQ       the same walk: S^T and dP^T = V dO^T, dQ^T += K^T dS^T with K in LDS; sums merged.
//   dK/dV    a workgroup owns 32 keys, one per lane; Q and dO blocks in LDS (row and transposed
//            fragments).  It forms each query block's row sums dO . O itself, so it waits for
//            nobody: no workspace, no flags, nothing to hand over between workgroups.
// All three form the scores from f16(Q * scale * log2e), as the 128-row kernels do.  Partial sums
// are added in wave order: results are reproducible bit for bit.
#include "common.h"

#include <algorithm>

namespace deers {

namespace {

template <int D>
struct SplitCfg {
  static constexpr int KS = D / 16;         // contraction steps over D
  static constexpr int DB = D / 32;         // 32-wide blocks of D
  static constexpr int RB = 2 * D;          // bytes per row
  static constexpr int CH = D / 8;          // 16-byte chunks per row
  static constexpr int BB = 32 * RB;        // bytes of a 32-row block
  static constexpr int NI = BB / 1024;      // loads per block
  static constexpr int kRound = DB > 2 ? 4 : 2 * DB;  // 16-column units merged per round
};

// Every load of this wave has landed, those into LDS included; LDS reads stay behind it.
__device__ __forceinline__ void settle_loads() {
  wait_all_vmem();
  asm volatile("" ::: "memory");
}

// Requests rows r0 .. r0 + 31 (rows past T - 1 read row T - 1) of a [T, D] matrix into the 32-row
// block at LDS address `dst`: 16-byte chunks, swizzled.
template <int D>
__device__ __forceinline__ void split_load_block(const half_t* base, int row_stride, int r0, int T, uint32_t dst,
                                                 int lane) {
  using C = SplitCfg<D>;
  constexpr int RPL = 1024 / C::RB;  // rows per load
  const int lane_row = lane / C::CH;
  if (r0 + 32 <= T) {  // the row of a load goes into its scalar base
    const uint32_t row_off = opaque((uint32_t)lane_row * (uint32_t)row_stride * 2);
    const half_t* row = base + (int64_t)r0 * row_stride;
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
      async_load16_to_lds(row + (int64_t)(i * RPL) * row_stride,
                          row_off + 16 * ((lane % C::CH) ^ lds_swizzle<C::CH>(i * RPL + lane_row)), dst, i * 1024);
  } else {
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
      async_load16_to_lds(base, (uint32_t)min(r0 + i * RPL + lane_row, T - 1) * (uint32_t)row_stride * 2 +
                                    16 * ((lane % C::CH) ^ lds_swizzle<C::CH>(i * RPL + lane_row)), dst, i * 1024);
  }
}

// Fragment ks of row lane % 32 (halfs 16 ks + 8 g ..) from a swizzled block in LDS.
template <int D>
__device__ __forceinline__ half8 split_row_frag(uint32_t block, int ks, int lane) {
  using C = SplitCfg<D>;
  const int r = lane & 31, g = lane >> 5;
  return lds_read_half8_at(block + r * C::RB + (((2 * ks + g) ^ lds_swizzle<C::CH>(r)) << 4));
}
// Transposed fragment: column 32 db + lane % 32, rows 16 ms + {4g .. 4g+3, 8+4g .. 8+4g+3}, the
// order in which registers 8 ms .. 8 ms + 7 of an accumulator hold their rows.
template <int D>
__device__ __forceinline__ half8 split_col_frag(uint32_t block, int ms, int db, int lane) {
  using C = SplitCfg<D>;
  const int g = lane >> 5, c4 = lane & 3;
  const int lrow = 4 * g + ((lane & 15) >> 2);
  const int chunk = 4 * db + 2 * ((lane >> 4) & 1) + (c4 >> 1);
  const uint32_t at = block + 16 * ms * C::RB + (c4 & 1) * 8;
  const half4 lo = lds_read_tr16_at(at + lrow * C::RB + ((chunk ^ lds_swizzle<C::CH>(lrow)) << 4));
  const half4 hi = lds_read_tr16_at(at + (lrow + 8) * C::RB + ((chunk ^ lds_swizzle<C::CH>(lrow + 8)) << 4));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// The KS fragments of row `row` of a [T, D] matrix from global memory.
template <int D>
__device__ __forceinline__ void split_global_frags(half8* f, const half_t* base, int row_stride, int row, int g) {
  const half_t* p = base + (int64_t)row * row_stride + 8 * g;
#pragma unroll
  for (int ks = 0; ks < SplitCfg<D>::KS; ++ks) f[ks] = *(const half8*)(p + 16 * ks);
}
template <int KS>
__device__ __forceinline__ void scale_frags(half8* f, float c) {
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e) f[ks][e] = (half_t)((float)f[ks][e] * c);
}
template <int KS>
__device__ __forceinline__ float dot_frags(const half8* a, const half8* b) {
  float s = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e) s = fmaf((float)a[ks][e], (float)b[ks][e], s);
  return pair_sum(s);
}
__device__ __forceinline__ half8 pack_regs(const floatx16& a, int ms) {
  half8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (half_t)a[8 * ms + e];
  return r;
}

// Adds the W waves' accumulators of a [32 rows, D] result (row = lane % 32, register r of block db
// is column 32 db + 8 (r / 4) + 4 g + r % 4), each scaled by its wave's `weight` first, in wave
// order, multiplies by `mul` and writes f16 rows at dst (this lane's row; not where !store).
// `red` is LDS for W * kRound * 8 * 64 floats.  Starts and ends with a barrier.
template <int D, int W>
__device__ __forceinline__ void merge_store(const floatx16* acc, float weight, float mul, half_t* dst, bool store,
                                            float* red, int wave, int lane) {
  using C = SplitCfg<D>;
  constexpr int R = C::kRound;
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int u0 = 0; u0 < 2 * C::DB; u0 += R) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R * 8; ++r)
      red[(wave * R * 8 + r) * 64 + lane] = acc[(u0 * 8 + r) / 16][(u0 * 8 + r) % 16] * weight;
    __syncthreads();
    for (int u = wave; u < R; u += W) {
      half4 x, y;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float s = red[(u * 8 + e) * 64 + lane];
#pragma unroll
        for (int w = 1; w < W; ++w) s += red[(w * R * 8 + u * 8 + e) * 64 + lane];
        if (e < 4) x[e & 3] = (half_t)(s * mul);
        else y[e & 3] = (half_t)(s * mul);
      }
      // the lane pair (l, l ^ 32) trades halves so that each stores 16 contiguous bytes
      const u32x2 xu = __builtin_bit_cast(u32x2, x), yu = __builtin_bit_cast(u32x2, y);
      const auto r0 = __builtin_amdgcn_permlane32_swap(xu[0], yu[0], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(xu[1], yu[1], false, false);
      if (store) *(u32x4*)(dst + 16 * (u0 + u) + 8 * (lane >> 5)) = u32x4{r0[0], r1[0], r0[1], r1[1]};
    }
  }
  __syncthreads();
}

template <int D, int W>
constexpr size_t merge_bytes() { return (size_t)W * SplitCfg<D>::kRound * 8 * 64 * sizeof(float); }

// ---- forward ----

// KREGS: the wave's next K fragments wait in registers, straight from global memory, and V has two
// blocks in LDS: the shortest stage.  Otherwise K and V have one block each in LDS, filled by whole
// cache lines and asked for again as soon as they have been read: half the LDS and a quarter of the lines
// per load, for launches in which several waves of a SIMD cover each other's waits.
template <int D, int W, bool KREGS>
constexpr size_t split_fwd_lds() {  // two blocks per wave, or the merge; then m and l of every wave
  return std::max((size_t)W * 2 * SplitCfg<D>::BB, merge_bytes<D, W>()) + W * 32 * 2 * sizeof(float);
}

template <int D, int W, bool KREGS>
__global__ __launch_bounds__(64 * W, 2) void attn_fwd_f16_split_kernel(FwdParams p, int BH, int n_blocks) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, T = p.T;
  int bh, rank;
  if (!map_block_even(blockIdx.x, n_blocks, BH, &bh, &rank)) return;
  const int qb = n_blocks - 1 - rank;  // longest rows first
  const int b_ = bh / p.H, h_ = bh % p.H;
  const half_t* K = (const half_t*)p.k + b_ * p.sk.b + h_ * p.sk.h;
  const half_t* V = (const half_t*)p.v + b_ * p.sv.b + h_ * p.sv.h;
  const int skt = (int)p.sk.t, svt = (int)p.sv.t;
  const int qrow = 32 * qb + (lane & 31);
  const uint32_t ring = lds_address(smem) + wave * 2 * C::BB;
  const uint32_t k_blk = ring + C::BB;
  uint32_t v_blk = ring;

  half8 kf[KREGS ? KS : 1], qf[KS];
  int kb = wave;
  auto request_k = [&](int block) {
    if constexpr (KREGS)
      split_global_frags<D>(kf, K, skt, min(32 * block + (lane & 31), T - 1), g);
    else
      split_load_block<D>(K, skt, 32 * block, T, k_blk, lane);
  };
  if (kb <= qb) {
    if (KREGS) split_load_block<D>(V, svt, 32 * kb, T, v_blk, lane);
    request_k(kb);
  }
  split_global_frags<D>(qf, (const half_t*)p.q + b_ * p.sq.b + h_ * p.sq.h, (int)p.sq.t, min(qrow, T - 1), g);
  if (!KREGS && kb <= qb) split_load_block<D>(V, svt, 32 * kb, T, v_blk, lane);
  if (!KREGS) wait_all_vmem();
  scale_frags<KS>(qf, p.scale_log2);

  floatx16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = ZERO16;
  float m = -INFINITY, l = 0.f;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    if constexpr (KREGS)
      settle_loads();  // K and V of this block
    else
      wait_vmcnt<C::NI>();  // K; V's block may be on its way
    floatx16 s = ZERO16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      half8 k;
      if constexpr (KREGS) k = kf[ks];
      else k = split_row_frag<D>(k_blk, ks, lane);
      s = mfma_f16(k, qf[ks], s);
    }
    if (more) {  // the next block's, under this block's work
      if constexpr (KREGS)
        split_load_block<D>(V, svt, 32 * (kb + W), T, v_blk ^ C::BB, lane);
      else
        settle_lds_reads();
      request_k(kb + W);
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
    if (__any(m_new > m)) {
      const float alpha = fast_exp2(m - m_new);  // 0 in the first block
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
      m = m_new;
    }
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - m);
      sum[r & 1] += s[r];
    }
    l += sum[0] + sum[1];
    if constexpr (!KREGS) {
      if (more)
        wait_vmcnt<C::NI>();  // V
      else
        wait_vmcnt<0>();
    }
#pragma unroll
    for (int ms = 0; ms < 2; ++ms) {
      const half8 pf = pack_regs(s, ms);
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] = mfma_f16(split_col_frag<D>(v_blk, ms, db, lane), pf, oacc[db]);
    }
    if constexpr (KREGS) {
      v_blk ^= C::BB;
    } else if (more) {
      settle_lds_reads();
      split_load_block<D>(V, svt, 32 * (kb + W), T, v_blk, lane);
    }
  }

  // ---- the waves' (m, l, O) become one; a wave without a block has m = -inf and weight 0 ----
  float* stat_m = (float*)(smem + split_fwd_lds<D, W, KREGS>() - W * 32 * 2 * sizeof(float));
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
  half_t* orow = (half_t*)p.o + b_ * p.so.b + h_ * p.so.h + (int64_t)min(qrow, T - 1) * p.so.t;
  merge_store<D, W>(oacc, fast_exp2(m - M), 1.f / L, orow, qrow < T, (float*)smem, wave, lane);
  if (wave == 0 && g == 0 && qrow < T) p.lse[(int64_t)bh * T + qrow] = (M + fast_log2(L)) * kLn2;
}

// ---- backward ----

template <int D, int W>
constexpr size_t split_bwd_lds() {  // two blocks of two operands per wave (or the merge), row statistics
  const size_t ring = (size_t)W * 4 * SplitCfg<D>::BB;
  return std::max(ring, merge_bytes<D, W>()) + W * 32 * 2 * sizeof(float);
}

template <int D, int W>
__device__ __forceinline__ void split_dq_body(const BwdParams& p, int bh, int qb, char* smem, int wave, int lane) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB;
  const int g = lane >> 5, T = p.T;
  const int b_ = bh / p.H, h_ = bh % p.H;
  const half_t* K = (const half_t*)p.k + b_ * p.sk.b + h_ * p.sk.h;
  const half_t* V = (const half_t*)p.v + b_ * p.sv.b + h_ * p.sv.h;
  const int skt = (int)p.sk.t, svt = (int)p.sv.t;
  const int qrow = 32 * qb + (lane & 31), qread = min(qrow, T - 1);
  const uint32_t ring = lds_address(smem) + wave * 4 * C::BB;

  half8 vf[KS], qf[KS], dof[KS];
  int kb = wave;
  if (kb <= qb) {
    split_load_block<D>(K, skt, 32 * kb, T, ring, lane);
    split_global_frags<D>(vf, V, svt, min(32 * kb + (lane & 31), T - 1), g);
  }
  float nd;
  {
    half8 of[KS];
    split_global_frags<D>(of, (const half_t*)p.o + b_ * p.so.b + h_ * p.so.h, (int)p.so.t, qread, g);
    split_global_frags<D>(dof, (const half_t*)p.d_o + b_ * p.sdo.b + h_ * p.sdo.h, (int)p.sdo.t, qread, g);
    split_global_frags<D>(qf, (const half_t*)p.q + b_ * p.sq.b + h_ * p.sq.h, (int)p.sq.t, qread, g);
    nd = -dot_frags<KS>(of, dof);
  }
  const float lse2 = -p.lse[(int64_t)bh * T + qread] * kLog2e;
  scale_frags<KS>(qf, p.scale_log2);

  floatx16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[db] = ZERO16;
  for (uint32_t slot = 0; kb <= qb; kb += W, slot ^= C::BB) {
    settle_loads();
    floatx16 s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = lse2;
      dp[r] = nd;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma_f16(split_row_frag<D>(ring + slot, ks, lane), qf[ks], s);
      dp = mfma_f16(vf[ks], dof[ks], dp);
    }
    if (kb + W <= qb) {
      split_load_block<D>(K, skt, 32 * (kb + W), T, ring + (slot ^ C::BB), lane);
      split_global_frags<D>(vf, V, svt, min(32 * (kb + W) + (lane & 31), T - 1), g);
    }
    if (kb == qb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r]) * dp[r];
#pragma unroll
    for (int ms = 0; ms < 2; ++ms) {
      const half8 ds = pack_regs(s, ms);
#pragma unroll
      for (int db = 0; db < DB; ++db) dq[db] = mfma_f16(split_col_frag<D>(ring + slot, ms, db, lane), ds, dq[db]);
    }
  }
  half_t* row = (half_t*)p.dq + b_ * p.sdq.b + h_ * p.sdq.h + (int64_t)qread * p.sdq.t;
  merge_store<D, W>(dq, 1.f, p.scale, row, qrow < T, (float*)smem, wave, lane);
}

template <int D, int W>
__device__ __forceinline__ void split_dkdv_body(const BwdParams& p, int bh, int kb, int n_blocks, char* smem, int wave,
                                                int lane) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB;
  const int g = lane >> 5, T = p.T;
  const int b_ = bh / p.H, h_ = bh % p.H;
  const half_t* Q = (const half_t*)p.q + b_ * p.sq.b + h_ * p.sq.h;
  const half_t* O = (const half_t*)p.o + b_ * p.so.b + h_ * p.so.h;
  const half_t* dO = (const half_t*)p.d_o + b_ * p.sdo.b + h_ * p.sdo.h;
  const float* lse = p.lse + (int64_t)bh * T;
  const int sqt = (int)p.sq.t, sot = (int)p.so.t, sdot = (int)p.sdo.t;
  const int krow = 32 * kb + (lane & 31), kread = min(krow, T - 1);
  const uint32_t ring = lds_address(smem) + wave * 4 * C::BB;
  float* stat = (float*)(smem + split_bwd_lds<D, W>() - W * 32 * 2 * sizeof(float)) + wave * 64;

  half8 of[KS], kf[KS], vf[KS];
  float lse_row = 0.f;
  int qb = kb + wave;
  auto request = [&](int block, uint32_t slot) {
    split_load_block<D>(Q, sqt, 32 * block, T, ring + slot, lane);
    split_load_block<D>(dO, sdot, 32 * block, T, ring + slot + C::BB, lane);
    const int row = min(32 * block + (lane & 31), T - 1);
    split_global_frags<D>(of, O, sot, row, g);
    lse_row = lse[row];
  };
  if (qb < n_blocks) request(qb, 0);
  split_global_frags<D>(kf, (const half_t*)p.k + b_ * p.sk.b + h_ * p.sk.h, (int)p.sk.t, kread, g);
  split_global_frags<D>(vf, (const half_t*)p.v + b_ * p.sv.b + h_ * p.sv.h, (int)p.sv.t, kread, g);

  floatx16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dk[db] = dv[db] = ZERO16;
  for (uint32_t slot = 0; qb < n_blocks; qb += W, slot ^= 2 * C::BB) {
    settle_loads();
    const uint32_t q_blk = ring + slot, do_blk = q_blk + C::BB;
    half8 dof[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) dof[ks] = split_row_frag<D>(do_blk, ks, lane);
    // the block's row statistics, one row per lane, to the rows the accumulators hold
    const float nd = -dot_frags<KS>(of, dof);
    const bool live = 32 * qb + (lane & 31) < T;  // a padded query's probabilities are zero
    if (g == 0) {
      stat[lane] = live ? -lse_row * kLog2e : -INFINITY;
      stat[32 + lane] = nd;
    }
    floatx16 s, dp;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 a = *(const floatx4*)(stat + 8 * r4 + 4 * g), b = *(const floatx4*)(stat + 32 + 8 * r4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * r4 + e] = a[e];
        dp[4 * r4 + e] = b[e];
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      half8 qs = split_row_frag<D>(q_blk, ks, lane);
      scale_frags<1>(&qs, p.scale_log2);
      s = mfma_f16(qs, kf[ks], s);
      dp = mfma_f16(dof[ks], vf[ks], dp);
    }
    if (qb + W < n_blocks) request(qb + W, slot ^ (2 * C::BB));
    if (qb == kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) < (lane & 31)) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r]);
      dp[r] *= s[r];
    }
#pragma unroll
    for (int ms = 0; ms < 2; ++ms) {
      const half8 pf = pack_regs(s, ms), ds = pack_regs(dp, ms);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        dv[db] = mfma_f16(split_col_frag<D>(do_blk, ms, db, lane), pf, dv[db]);
        dk[db] = mfma_f16(split_col_frag<D>(q_blk, ms, db, lane), ds, dk[db]);
      }
    }
  }
  half_t* dv_row = (half_t*)p.dv + b_ * p.sdv.b + h_ * p.sdv.h + (int64_t)kread * p.sdv.t;
  half_t* dk_row = (half_t*)p.dk + b_ * p.sdk.b + h_ * p.sdk.h + (int64_t)kread * p.sdk.t;
  merge_store<D, W>(dv, 1.f, 1.f, dv_row, krow < T, (float*)smem, wave, lane);
  merge_store<D, W>(dk, 1.f, p.scale, dk_row, krow < T, (float*)smem, wave, lane);
}

// Ranks alternate between the roles, longest first: rank 2 r is the dK/dV block of keys 32 r ..,
// rank 2 r + 1 the dQ block as many rows from the end.
template <int D, int W>
__global__ __launch_bounds__(64 * W, D == 128 ? 1 : 2) void attn_bwd_f16_split_kernel(BwdParams p, int BH, int n_blocks) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, rank;
  if (!map_block_even(blockIdx.x, 2 * n_blocks, BH, &bh, &rank)) return;
  if (rank & 1)
    split_dq_body<D, W>(first_argument<BwdParams>(), bh, n_blocks - 1 - (rank >> 1), smem, wave, lane);
  else
    split_dkdv_body<D, W>(first_argument<BwdParams>(), bh, rank >> 1, n_blocks, smem, wave, lane);
}

template <int D, int W, bool KREGS>
void launch_fwd_split(const FwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_fwd_f16_split_kernel<D, W, KREGS>;
  constexpr size_t lds = split_fwd_lds<D, W, KREGS>();
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  hipLaunchKernelGGL(kernel, dim3(map_even_blocks(n_blocks, BH)), dim3(64 * W), lds, stream, p, BH, n_blocks);
}
template <int D, int W>
void launch_bwd_split(const BwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_bwd_f16_split_kernel<D, W>;
  constexpr size_t lds = split_bwd_lds<D, W>();
  static bool attr_set = false;
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  hipLaunchKernelGGL(kernel, dim3(map_even_blocks(2 * n_blocks, BH)), dim3(64 * W), lds, stream, p, BH, n_blocks);
}

}  // namespace

// Which launches come here and in which form, measured on T = 32 .. 8192, 3 .. 800 heads and the three
// head widths against the 128-row kernels and between 1, 2 and 4 waves.  nb = T / 32 is the length of a
// walk, n = heads * nb the number of workgroups, u = n * D / 64 their number weighted by what a block
// of the other operand weighs.
//
// Waves: four while the workgroups are few, and for long walks (forward D = 64, us in 4 / 2 / 1 waves:
// 12 x 512 6.8 / 9.2 / 13.7, 24 x 1024 11.0 / 15.1 / 24.9, 96 x 256 7.3 / 7.1 / 9.1; backward 12 x 512
// 11 / 12 / 18, 384 x 64 17 / 13 / 10); never more than blocks to walk.  KREGS where one wave per SIMD is
// all there is, and at head width 32, whose fragments are two loads (3 x 4096 x 32 15.1 us against 19.2,
// 12 x 256 x 64 5.5 against 6.0, 24 x 1024 x 64 14.3 against 11.0).
//
// Takes, 128-row kernels -> these: short walks gain throughout, what the others do for 128 rows that
// are not there (forward 800 x 64 x 64 10.2 -> 7.2, 384 x 256 x 64 13.8 -> 12.9; backward 384 x 64 x 64 16.0 -> 10.2,
// 384 x 256 x 32 24.1 -> 18.9).  Longer walks gain while the device is not full: forward 15 x 777 x 128 18.3 ->
// 12.6, 36 x 1024 x 64 17.4 -> 16.2, 16 x 2048 x 128 38.7 -> 36.7 (48 x 1024 x 64 18.1 -> 18.5); backward, which streams
// three operands per block, 3 x 4096 x 64 86 -> 47, 12 x 1024 x 64 24.1 -> 21.4, 24 x 400 x 128 25.5 -> 21.4 (16 x 2048 x
// 64 36.4 -> 37.6, 24 x 1024 x 64 27.6 -> 27.7).  The backward's line at head width 128, 128-row kernels / these, us,
// u in parentheses: below 28 blocks 24 x 512 (768) 27.7 / 23.0, 16 x 768 (768) 32.7 / 29.4, 18 x 700 (792, in four
// waves) 31.3 / 47.6; from 28 on 11 x 896 (616) 35.0 / 32.8, 12 x 896 (672) 35.2 / 36.5, 9 x 1024 (576) 37.0 / 32.9,
// 11 x 1024 (704) 37.3 / 38.8, 8 x 1280 (640) 42.7 / 46.2; from 48 on 7 x 1536 (672) 48.5 / 47.5, 8 x 1536 (768) 49.2 / 56.9,
// 6 x 2048 (768) 60.3 / 63.7, 4 x 3072 (768) 87.3 / 93.9; from 128 on 3 x 4096 (768) 171 / 106, 2 x 6144 (768) 247 / 167.
struct SplitSize {
  int64_t nb, u;
  SplitSize(int64_t BH, int64_t T, int64_t D) : nb((T + 31) / 32), u(BH * nb * D / 64) {}
};
bool attn_fwd_f16_split_takes(int64_t BH, int64_t T, int64_t D) {
  const SplitSize z(BH, T, D);
  return z.nb <= 8 ? z.u <= 3200 : z.u <= (D == 128 ? 2048 : 1200);
}
bool attn_bwd_f16_split_takes(int64_t BH, int64_t T, int64_t D) {
  const SplitSize z(BH, T, D);
  if (D == 128 && z.nb > 8) return z.u <= (z.nb < 28 || z.nb >= 128 ? 768 : z.nb < 48 ? 624 : 672);
  return z.u <= (z.nb <= 4 ? 3200 : z.nb <= 8 ? 1600 : z.nb <= 16 ? 768 : 448);
}
static int fwd_waves(const SplitSize& z) {
  const int64_t most = z.u <= 320 ? z.nb : z.u <= 1200 ? z.nb / 2 : z.nb / 4;
  const int64_t w = z.u <= 640 || (z.nb >= 16 && z.u <= 1152) || z.nb >= 64 ? 4 : z.u <= 1536 ? 2 : 1;
  return (int)std::min(w, most);
}
static int bwd_waves(const SplitSize& z) {
  const int64_t w = z.u <= 256 || z.nb >= 28 ? 4 : z.u <= (z.nb <= 8 ? 512 : 768) ? 2 : 1;
  return (int)std::min(w, z.u <= 256 ? z.nb : z.nb / 4);
}

template <int D, int W>
static void launch_fwd(const FwdParams& p, int BH, bool kregs, hipStream_t stream) {
  if constexpr (D != 32) {
    if (!kregs) return launch_fwd_split<D, W, false>(p, BH, stream);
  }
  launch_fwd_split<D, W, true>(p, BH, stream);
}
template <int D>
static void launch_fwd(const FwdParams& p, int BH, hipStream_t stream) {
  const SplitSize z(BH, p.T, D);
  const int w = fwd_waves(z);
  const bool kregs = z.u <= 192;
  if (w >= 4)
    launch_fwd<D, 4>(p, BH, kregs, stream);
  else if (w >= 2)
    launch_fwd<D, 2>(p, BH, kregs, stream);
  else
    launch_fwd<D, 1>(p, BH, kregs, stream);
}
template <int D>
static void launch_bwd(const BwdParams& p, int BH, hipStream_t stream) {
  const int w = bwd_waves(SplitSize(BH, p.T, D));
  if (w >= 4)
    launch_bwd_split<D, 4>(p, BH, stream);
  else if (w >= 2)
    launch_bwd_split<D, 2>(p, BH, stream);
  else
    launch_bwd_split<D, 1>(p, BH, stream);
}

void launch_attn_fwd_f16_split(const FwdParams& p, int B, int D, hipStream_t stream) {
  LaunchScope scope("attn_fwd_f16", stream);
  switch (D) {
    case 32: launch_fwd<32>(p, B * p.H, stream); break;
    case 64: launch_fwd<64>(p, B * p.H, stream); break;
    case 128: launch_fwd<128>(p, B * p.H, stream); break;
  }
}
void launch_attn_bwd_f16_split(const BwdParams& p, int B, int D, hipStream_t stream) {
  LaunchScope scope("attn_bwd_f16", stream);
  switch (D) {
    case 32: launch_bwd<32>(p, B * p.H, stream); break;
    case 64: launch_bwd<64>(p, B * p.H, stream); break;
    case 128: launch_bwd<128>(p, B * p.H, stream); break;
  }
}

}  // namespace deers
