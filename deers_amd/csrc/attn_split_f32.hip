// Fused causal attention of up to middling launches, f32 storage and arithmetic, gfx950: forward and
// backward of the same contract as attn_fwd_f32.hip and attn_bwd_f32.hip
// (src/models/gpt.rs:139-144; src/ops.rs:1089-1101, 422-425, 210-214, 777-799, 1162-1175, 638-643).
//
// The forward of attn_fwd_f32.hip gives a workgroup 128 rows whose four waves walk the other operand
// together, a chain of T / 32 stages with barriers.  Here a workgroup owns 32 rows and its W waves
// divide the 32-row blocks of the other operand (wave w takes blocks w, w + W, ...), without a barrier
// until their partial sums meet at the end, so the chain of a wave is T / (32 W) stages and four times
// as many workgroups are in flight.
//
//   forward  S^T = K Q^T, O^T += V^T P^T; online softmax per wave; O, m and l are merged.
//   dQ       dP^T = V dO^T, S^T, dQ^T += K^T dS^T; sums merged.
//   dK/dV    a workgroup owns 32 keys: dP = dO V^T, S = Q K^T, dV^T += dO^T P, dK^T += Q^T dS.  It forms
//            each query block's row sums dO . O itself: no workspace, no hand-over.
// The backward computes S and dP twice, 7 products per block against the 5 of attn_bwd_f32.hip: the
// price of one launch whose workgroups wait for nobody.  Partial sums are added in wave order:
// dQ, dK and dV are reproducible bit for bit.
//
// A wave's first loads and its merge cost it some 10 K clocks; blocks are dealt so that every XCD has
// the same number of them also when the heads are not a multiple of eight (map_block_even), and, while all are resident
// at once, so that the CUs have even totals (paired_block; 24 x 256 x 32 backward 11.3 -> 10.3 us, 12 x 512 x 32 17.4 ->
// 14.4, forward 24 x 512 x 64 17.9 -> 14.3; not at head width 128, where one workgroup fills a CU and the index
// arithmetic costs the forward 6 %).
//
// A product costs 64 clocks of matrix pipe per two elements of D (v_mfma_f32_32x32x2_f32), so the
// pipe is the bound as long as a wave's blocks arrive in time.  The operand whose block is asked for
// last is the one that the next stage needs second, so that both requests are covered by a product
// (2048 clocks at D = 64).
//
// us, forward / backward, 128-row kernels -> these: 24 heads x 256 x 32 15.6 / 26.9 -> 5.8 / 10.1, 12 x 512 x 64
// 41 / 66 -> 14 / 32, 12 x 1024 x 64 77 / 119 -> 23 / 67, 3 x 4096 x 32 191 / 337 -> 55 / 129, 8 x 256 x 128 48 / 98
// -> 15 / 29.
#include <algorithm>

#include "attn_f32_blocks.h"

namespace deers {

namespace {

// ---- forward ----

template <int D, int W>
__global__ __launch_bounds__(64 * W, Split32<D>::kWavesPerSimd) void attn_fwd_f32_split_kernel(FwdParams p, int BH, int n_blocks, int cus) {
  fetch_arguments<decltype(attn_fwd_f32_split_kernel<D, W>)>();
  using C = Split32<D>;
  constexpr int KH = C::KH, DB = C::DB;
  // More than 256 registers in all, so that a SIMD takes one wave: with 208 a CU's workgroups of one or two waves come to lie two
  // on a SIMD, beside idle ones (12 heads x 2094 x 128 227 us, 149 so; 48 x 1024 197 / 136).
  if constexpr (D == 128) asm volatile("" ::: "a63");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, T = p.T;
  int bh, rank;
  if (!map_block_even(D == 128 ? blockIdx.x : paired_block(blockIdx.x, gridDim.x, cus), n_blocks, BH, &bh, &rank)) return;
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

  floatx16 oacc[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[0][db] = ZERO16;
  // The reference m of a row's exponentials is the maximum of its first block, and moves when a later
  // score exceeds it by more than 2^8: `ref` is -m in the layout of the products, which start from it, so
  // that the usual stage has no subtraction and no rescaling (some 60 of 110 vector instructions).
  // At head width 128 the sums live in accumulation registers, and a branch around them copies them.
  constexpr bool kLazy = D < 128;
  const bool any = kb <= qb;
  bool first = true;
  floatx16 ref = ZERO16;
  float m = kLazy ? 0.f : -INFINITY, l = 0.f;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    wait_vmcnt<C::NI>();  // K; V's block may be on its way
    floatx16 s = product<D>(k_blk, qf, ref, lane);
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
    const float top = pair_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
    if (!kLazy || first || __any(top > 8.f)) {
      const float m_new = kLazy ? m + (first ? top : fmaxf(top, 0.f)) : fmaxf(m, top);
      // the first block's scales zeros: by no more than one, where all of its scores lie far below zero
      const float alpha = fast_exp2(fminf(m - m_new, 0.f));
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[0][db] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] -= kLazy ? m_new - m : m_new;
        if (kLazy) ref[r] = -m_new;
      }
      m = m_new;
      first = false;
    }
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r]);
      sum[r & 1] += s[r];
    }
    l += sum[0] + sum[1];
    if (more)
      wait_vmcnt<C::NI>();  // V
    else
      wait_vmcnt<0>();
    accumulate<D>(oacc[0], v_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(V, svt, 32 * (kb + W), T, v_blk, lane);
    }
  }

  // ---- the waves' (m, l, O) become one; a wave without a block has m = -inf and weight 0 ----
  float* stat_m = split32_stats<D, W>(smem);
  float* stat_l = stat_m + W * 32;
  l = pair_sum(l);
  if (!any) m = -INFINITY;
  if (g == 0) {
    stat_m[wave * 32 + lane] = m;
    stat_l[wave * 32 + lane] = l;
  }
  settle_lds_reads();
  leave_sums<D, W, 1, 2 * C::BB>(oacc, k_blk, lane);
  float M = -INFINITY, L = 0.f, weight[W];
#pragma unroll
  for (int w = 0; w < W; ++w) M = fmaxf(M, stat_m[w * 32 + (lane & 31)]);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    weight[w] = fast_exp2(stat_m[w * 32 + (lane & 31)] - M);
    L += stat_l[w * 32 + (lane & 31)] * weight[w];
  }
  float* const orow = (float*)p.o + b * p.so.b + h * p.so.h + (int64_t)min(qrow, T - 1) * p.so.t;
  const float inv = 1.f / L;
  store_sums<D, W, 1, 2 * C::BB, true>(oacc, lds_address(smem), weight, &inv, &orow, qrow < T, wave, lane);
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

  floatx16 dq[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[0][db] = ZERO16;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    wait_vmcnt<C::NI>();  // V; K's block may be on its way
    // (from zero, not from the row statistics: see the error figures in attn_bwd_f32.hip)
    const floatx16 dp = product<D>(v_blk, dof, ZERO16, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(V, svt, 32 * (kb + W), T, v_blk, lane);
      wait_vmcnt<C::NI>();  // K
    } else {
      wait_vmcnt<0>();
    }
    floatx16 s = product<D>(k_blk, qf, ZERO16, lane);
    if (kb == qb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r] + lse2) * (dp[r] + nd);
    accumulate<D>(dq[0], k_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(K, skt, 32 * (kb + W), T, k_blk, lane);
    }
  }
  float* const row = (float*)p.dq + b * p.sdq.b + h * p.sdq.h + (int64_t)qread * p.sdq.t;
  const float mul = p.scale;
  settle_lds_reads();
  leave_sums<D, W, 1, 2 * C::BB>(dq, k_blk, lane);
  store_sums<D, W, 1, 2 * C::BB>(dq, lds_address(smem), nullptr, &mul, &row, qrow < T, wave, lane);
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
  float lse_row = lse[min(32 * qb + (lane & 31), T - 1)];
  if (qb < n_blocks) {
    load_block<D>(Q, sqt, 32 * qb, T, q_blk, lane);
    load_block<D>(dO, sdot, 32 * qb, T, do_blk, lane);
  }
  wait_all_vmem();
#pragma unroll
  for (int k = 0; k < KH; ++k) kf[k] *= p.scale_log2;

  floatx16 acc[2][DB];  // dK, dV
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = acc[1][db] = ZERO16;
  for (; qb < n_blocks; qb += W) {
    const bool more = qb + W < n_blocks;
    const int row = 32 * qb + (lane & 31), read = min(row, T - 1);
    float of[KH], sum;
    row_frag<D>(of, O, p.so.t, read, g);  // used under the second product
    if (g == 0) stat[lane] = row < T ? -lse_row * kLog2e : -INFINITY;  // a padded query's probabilities are zero
    wait_vmcnt<2 * C::NI>();  // Q; dO's block may be on its way
    // (the statistics later: as the first product's accumulator they would be waited for)
    floatx16 s = product<D>(q_blk, kf, ZERO16, lane);
    wait_vmcnt<C::NI>();  // dO
    floatx16 dp = product<D, true>(do_blk, vf, ZERO16, lane, of, &sum);
    sum = pair_sum(sum);
    if (g == 0) stat[32 + lane] = -sum;
    if (qb == kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) < (lane & 31)) s[r] = -INFINITY;
    }
    const floatx16 d = stat_rows(stat + 32, g);
    s += stat_rows(stat, g);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r]);
      dp[r] = s[r] * (dp[r] + d[r]);
    }
    accumulate<D>(acc[0], q_blk, dp, lane);
    if (more) {
      settle_lds_reads();
      lse_row = lse[min(32 * (qb + W) + (lane & 31), T - 1)];
      load_block<D>(Q, sqt, 32 * (qb + W), T, q_blk, lane);
    }
    accumulate<D>(acc[1], do_blk, s, lane);
    if (more) {
      settle_lds_reads();
      load_block<D>(dO, sdot, 32 * (qb + W), T, do_blk, lane);
    }
  }
  float* const row[2] = {(float*)p.dk + b * p.sdk.b + h * p.sdk.h + (int64_t)kread * p.sdk.t,
                         (float*)p.dv + b * p.sdv.b + h * p.sdv.h + (int64_t)kread * p.sdv.t};
  const float mul[2] = {p.scale, 1.f};
  settle_lds_reads();
  leave_sums<D, W, 2, 2 * C::BB>(acc, q_blk, lane);
  store_sums<D, W, 2, 2 * C::BB>(acc, lds_address(smem), nullptr, mul, row, krow < T, wave, lane);
}

// Ranks alternate between the roles, longest first: rank 2 r is the dK/dV block of keys 32 r ..,
// rank 2 r + 1 the dQ block as many rows from the end.
template <int D, int W>
__global__ __launch_bounds__(64 * W, Split32<D>::kWavesPerSimd) void attn_bwd_f32_split_kernel(BwdParams p, int BH, int n_blocks, int cus) {
  fetch_arguments<decltype(attn_bwd_f32_split_kernel<D, W>)>();
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, rank;
  if (!map_block_even(D == 128 ? blockIdx.x : paired_block(blockIdx.x, gridDim.x, cus), 2 * n_blocks, BH, &bh, &rank)) return;
  if (rank & 1)
    split32_dq<D, W>(first_argument<BwdParams>(), bh, n_blocks - 1 - (rank >> 1), smem, wave, lane);
  else
    split32_dkdv<D, W>(first_argument<BwdParams>(), bh, rank >> 1, n_blocks, smem, wave, lane);
}

template <int D, int W>
void launch_fwd_split(const FwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_fwd_f32_split_kernel<D, W>;
  constexpr size_t lds = split32_lds<D, W>();
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  const int grid = map_even_blocks(n_blocks, BH);
  static PairedState paired;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * W), lds, stream, p, BH, n_blocks,
                     paired_cus(paired, kernel, 64 * W, lds, grid));
}
template <int D, int W>
void launch_bwd_split(const BwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_bwd_f32_split_kernel<D, W>;
  constexpr size_t lds = split32_lds<D, W>();
  static bool attr_set = false;
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  const int grid = map_even_blocks(2 * n_blocks, BH);
  static PairedState paired;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * W), lds, stream, p, BH, n_blocks,
                     paired_cus(paired, kernel, 64 * W, lds, grid));
}

}  // namespace

// Which launches come here and with how many waves per workgroup.  Measured on T = 32 .. 8192, 1 ..
// 4000 heads and the three head widths against the other kernels and between 1, 2 and 4 waves (the forward anew: 850
// launches; its rules are on average 0.4 % behind the best form); nb = T / 32 is the length of a walk, n = heads * nb the
// number of workgroups.
//
// Waves.  Few workgroups: four waves, the shortest chain (us in 4 / 2 / 1: 13 x 512 x 64 14 / 22 / 39, 25 x 4096 x 64 441 /
// 500 / 590).  Many: the SIMDs are covered anyway, and a wave that walks longer pays its start-up and its merge less often
// (168 x 400 x 128 132 / 97 / 83, 480 x 400 x 64 140 / 126 / 113); the shorter the walks, the fewer workgroups that takes, and the
// longer they are, the more are needed for the last ones to end together (in 4 / 1: 90 x 2395 x 32 269 / 296, 30 x 8192 x 32 988 /
// 1068).  Walks of up to 12 blocks were timed on a grid of their own: in 4 / 2 / 1 312 x 121 x 32 10.4 / 8.5 / 9.4, 235 x 89 x 32 7.3 / 5.9 / 6.9,
// 152 x 185 x 128 41.8 / 28.7 / 33.5, 258 x 57 x 128 25.3 / 17.7 / 14.5; a line at 256 or 512 is where the device's SIMDs have taken as many waves as
// they hold (122 x 123 x 64, 488 workgroups of four waves, 9.9 and of two 10.7).  At head width 128 a SIMD has one wave, so
// that two or one are enough early (65 x 1024 x 128 208 / 175 / 161).
//
// Takes, forward, us in the 128-row kernel / here: nearly everything, since that one forms 128 rows and has barriers
// where waves here wait for themselves only (100 x 1024 x 64 143 / 130, 25 x 4096 x 64 559 / 441, 168 x 400 x 128 119 / 83, 65 x 1024
// x 128 197 / 161, 25 x 4096 x 128 1137 / 928), up to the size where a four-fold reuse of K and V tiles decides (563 x
// 1024 x 64 705 / 717, 375 x 1024 x 128 950 / 963, 563 x 1024 x 128 1432 / 1583; shorter walks later).
extern bool attn_128_rows;  // runtime.hip
bool attn_f32_one_wave(int64_t n, int64_t nb, int64_t D) {
  return n >= (D == 32 ? 4608 + 48 * nb : D == 64 ? 1800 + 80 * nb : 1152 + 48 * nb);
}
bool attn_fwd_f32_split_takes(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (attn_128_rows) return D == 32;
  if (D == 32 || nb <= 8) return true;
  if (D == 128) return n <= (nb <= 10 ? 18000 : nb >= 13 && nb <= 15 ? 12000 : 9000);
  return n <= (nb <= 24 ? 20000 : 16000);
}
static int fwd_waves(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (nb < 2) return 1;
  int64_t four, two;  // workgroups up to which there are as many waves
  if (D == 32) {
    four = nb < 4 ? 350 : nb < 10 ? std::min(180 * nb, 560 + 66 * nb) : std::min<int64_t>(std::max<int64_t>(6500, 4608 + 48 * nb), 170 * nb - 150);
    two = nb < 3 ? 330 : nb < 10 ? std::min<int64_t>(350 * nb - 50, 2500) : nb < 12 && n > 230 * nb && n <= 3750 ? 0 : nb < 16 ? 5300 : 7000;
  } else if (D == 64) {
    four = nb < 4 ? 330 : nb < 5 ? (n > 440 ? 512 : 256) : nb < 8 ? std::min<int64_t>(110 * nb, 650) : nb < 9 ? 900 : nb < 12 ? 1100 : std::min(175 * nb - 560, 2600 + 36 * nb);
    two = nb < 3 ? 350 : nb < 4 ? 800 : nb < 11 ? std::min<int64_t>(200 * nb, 1800) : 3200;
  } else {
    four = nb < 9 ? std::max<int64_t>(60 * nb, 256) : std::max<int64_t>(510, 400 + 9 * nb);
    two = nb < 3 ? 512 : nb < 4 ? 800 : nb < 9 ? std::max<int64_t>(1000, 150 * nb) : nb < 12 ? 1300 : nb < 16 ? 1400 : nb >= 48 && n > 2200 ? 3400 : 1650;
  }
  return nb >= 3 && n <= four ? 4 : n <= two ? 2 : 1;
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
