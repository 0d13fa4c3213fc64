// Fused causal attention backward, f32 storage and arithmetic, gfx950: two passes with dS in memory
// (src/ops.rs:422-425, 210-214, 777-799, 1162-1175, 638-643).
//
//   prep    per query row -LSE*log2(e) and -rowsum(dO o O), padded.
//   dK/dV   a workgroup owns 32 keys, its W waves divide the 32-row query blocks at or below the diagonal
//           without a barrier until their sums meet: S = Q K^T, dP = dO V^T, P = exp2(S*scale*log2e + lse2),
//           dS = P o (dP - rowsum), dV^T += dO^T P, dK^T += Q^T dS; dS goes to memory, 4 KB per block.
//   dQ      a workgroup owns 32 queries, its waves divide the key blocks: dQ^T += K^T dS^T.
// Five products per block and no other work that counts, bound by the matrix pipe (a product of two
// 32 x D blocks is 64 D / 2 clocks, v_mfma_f32_32x32x2_f32, so a block costs the dK/dV pass 8.2 K clocks at
// D = 64).  4 KB of dS per 10.2 K clocks are a tenth of what memory takes.  What was tried instead of dS in
// memory, us at 24 heads x 4096 x 64 (the pipe alone: 920):
//   dQ by f32 atomics from the one pass: 1330.  The adds leave the XCD's L2 (every one is performed at the
//     memory side); without them the kernel took 950.
//   the same with 128 keys per workgroup in lockstep and their dQ summed through LDS first, a quarter of the
//     adds: 1160.  Kernels of that kind with swizzled LDS addresses stood here before: 1222.
//   S and dP computed again for dQ, 7 products (attn_split_f32.hip): better where the launch is small.
//   these: 1037 with products that started from the row statistics (below), 1060 now.
// Every sum is taken in a fixed order: dQ, dK and dV are reproducible bit for bit.
//
// The products start from zero and the row statistics are added to the finished sums.  Starting them from
// the statistics saves 32 additions per block (8 x 12 x 1024 x 64, forward and backward: 442 us, 446 this way)
// but rounds every element's term at the size of the LSE: relative error of dQ against 64 bits 1.0e-6 instead
// of 0.43e-6 at T = 1024, D = 64, of dK 1.06e-6 instead of 0.53e-6.
//
// us, kernels of that kind -> these: 8 x 12 x 1024 x 64 366 -> 305, 400 x 512 x 64 427 -> 352, 8 x 2048 x 64 162 -> 132, 48 x
// 1024 x 128 499 -> 370, 400 x 512 x 128 1225 -> 747, 96 x 1024 x 32 199 -> 168.
#include <algorithm>

#include "attn_f32_blocks.h"

namespace deers {

namespace {

// The row statistics as the dK/dV pass reads them, lse2 = -LSE*log2(e) and negdelta = -rowsum(dO o O), rows
// padded to t_pad per head (-inf and 0 there).  Reads O and dO once: 11 us for 96 x 1024 x 64, 4.5 TB/s.
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_prep_f32_kernel(BwdParams p, int64_t rows) {
  fetch_arguments<decltype(attn_bwd_prep_f32_kernel<D>)>();
  constexpr int LPR = D / 4;  // lanes per row, 16 bytes each
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;  // of [B*H][t_pad]
  const int part = threadIdx.x % LPR;
  if (row >= rows) return;
  const int bh = (int)(row / p.t_pad), t = (int)(row % p.t_pad);
  const int b = bh / p.H, h = bh % p.H;
  float acc = 0.f;
  if (t < p.T) {
    const floatx4 ov = *(const floatx4*)((const float*)p.o + b * p.so.b + h * p.so.h + t * p.so.t + 4 * part);
    const floatx4 dv = *(const floatx4*)((const float*)p.d_o + b * p.sdo.b + h * p.sdo.h + t * p.sdo.t + 4 * part);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc += ov[e] * dv[e];
  }
#pragma unroll
  for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (part == 0) {
    p.lse2[row] = t < p.T ? -p.lse[(int64_t)bh * p.T + t] * kLog2e : -INFINITY;
    p.negdelta[row] = t < p.T ? -acc : 0.f;
  }
}

// Bytes of one 32 x 32 block of dS and its number among a head's: a query block's are contiguous.  Inside
// a block the writer's registers as they are: 1 KB per four registers, 16 bytes per lane, whole cache lines.
constexpr int kDsBlock = 4096;
constexpr int kDsPitch = 1024 + 16;  // of a block's loads in LDS: four of eight query groups share no banks
__host__ __device__ __forceinline__ int64_t ds_block(int qb, int kb) { return (int64_t)qb * (qb + 1) / 2 + kb; }

template <int D, int W>
__global__ __launch_bounds__(64 * W, Split32<D>::kWavesPerSimd) void attn_bwd_f32_dkdv_kernel(BwdParams p, int bh0, int BH,
                                                                                         int n_blocks, char* ds) {
  fetch_arguments<decltype(attn_bwd_f32_dkdv_kernel<D, W>)>();
  using C = Split32<D>;
  constexpr int KH = C::KH, DB = C::DB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, kb;
  if (!map_block_even(blockIdx.x, n_blocks, BH, &bh, &kb)) return;
  bh = __builtin_amdgcn_readfirstlane(bh);
  kb = __builtin_amdgcn_readfirstlane(kb);
  char* ds_head = ds + (int64_t)bh * ds_block(n_blocks, 0) * kDsBlock;
  bh += bh0;
  const int g = lane >> 5, T = p.T;
  const int b = bh / p.H, h = bh % p.H;
  const float* Q = (const float*)p.q + b * p.sq.b + h * p.sq.h;
  const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
  const float* dO = (const float*)p.d_o + b * p.sdo.b + h * p.sdo.h;
  const int sqt = (int)p.sq.t, sdot = (int)p.sdo.t;
  const int krow = 32 * kb + (lane & 31), kread = min(krow, T - 1);
  const uint32_t q_blk = lds_address(smem) + wave * 2 * C::BB, do_blk = q_blk + C::BB;
  float* stat = split32_stats<D, W>(smem) + wave * 64;
  const uint32_t stat_lds = lds_address(stat);
  // lse2 and negdelta of a block's 32 rows: one 4-byte load per lane
  const float* stats = p.lse2 + (int64_t)bh * p.t_pad;
  const uint32_t stat_off = (lane & 31) * 4 + (g ? (uint32_t)((const char*)p.negdelta - (const char*)p.lse2) : 0u);

  int qb = kb + wave;
  if (qb < n_blocks) {
    async_load4_to_lds(stats + 32 * qb, stat_off, stat_lds);
    load_block<D>(Q, sqt, 32 * qb, T, q_blk, lane);
    load_block<D>(dO, sdot, 32 * qb, T, do_blk, lane);
  }
  float kf[KH], vf[KH];
  row_frag<D>(kf, K, p.sk.t, kread, g);
  row_frag<D>(vf, (const float*)p.v + b * p.sv.b + h * p.sv.h, p.sv.t, kread, g);
  wait_all_vmem();
#pragma unroll
  for (int k = 0; k < KH; ++k) kf[k] *= p.scale_log2;

  floatx16 acc[2][DB];  // dK, dV
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = acc[1][db] = ZERO16;
  for (; qb < n_blocks; qb += W) {
    const bool more = qb + W < n_blocks;
    wait_vmcnt<C::NI>();  // dS written, statistics, Q
    floatx16 s = product<D>(q_blk, kf, ZERO16, lane);
    wait_vmcnt<0>();  // dO
    floatx16 dp = product<D>(do_blk, vf, ZERO16, lane);
    s += stat_rows(stat, g);
    dp += stat_rows(stat + 32, g);
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
    {
      char* to = ds_head + ds_block(qb, kb) * kDsBlock;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *(floatx4*)(to + 1024 * r4 + (uint32_t)lane * 16) =
            floatx4{dp[4 * r4], dp[4 * r4 + 1], dp[4 * r4 + 2], dp[4 * r4 + 3]};
      asm volatile("" ::: "memory");
    }
    accumulate<D>(acc[0], q_blk, dp, lane);
    if (more) {
      settle_lds_reads();
      async_load4_to_lds(stats + 32 * (qb + W), stat_off, stat_lds);
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

// A wave of the dQ pass has one K block and one block of dS in LDS (12.5 KB at D = 64): three to a SIMD
// cover each other's waits better than fewer with two of each.
template <int D, int W>
struct DqPass {
  using C = Split32<D>;
  static constexpr int WAVE = C::BB + 4 * kDsPitch;
  static constexpr int LDS = W * WAVE;
};

template <int D, int W>
__global__ __launch_bounds__(64 * W) void attn_bwd_f32_dq_kernel(BwdParams p, int bh0, int BH, int n_blocks,
                                                                 const char* ds) {
  fetch_arguments<decltype(attn_bwd_f32_dq_kernel<D, W>)>();
  using C = Split32<D>;
  using S = DqPass<D, W>;
  constexpr int DB = C::DB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, rank;
  if (!map_block_even_by_search(blockIdx.x, n_blocks, BH, &bh, &rank)) return;
  bh = __builtin_amdgcn_readfirstlane(bh);
  const int qb = __builtin_amdgcn_readfirstlane(n_blocks - 1 - rank);  // longest rows first
  const char* ds_row = ds + ((int64_t)bh * ds_block(n_blocks, 0) + ds_block(qb, 0)) * kDsBlock;
  bh += bh0;
  const int g = lane >> 5, T = p.T;
  const int b = bh / p.H, h = bh % p.H;
  const float* K = (const float*)p.k + b * p.sk.b + h * p.sk.h;
  const int skt = (int)p.sk.t;
  const uint32_t lds = lds_address(smem) + wave * S::WAVE;
  // where the writer's lane (key) and register (query) have put the element of this lane's query and key 4 g
  const int q = lane & 31;
  const uint32_t ds_at = C::BB + (q >> 3) * kDsPitch + ((q >> 2) & 1) * 512 + (q & 3) * 4 + g * 64;

  floatx16 acc[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = ZERO16;
  for (int kb = wave; kb <= qb; kb += W) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      async_load16_to_lds(ds_row + (int64_t)kb * kDsBlock + 1024 * i, lane * 16, lds, C::BB + i * kDsPitch);
    load_block<D>(K, skt, 32 * kb, T, lds, lane);
    wait_vmcnt<0>();
    floatx16 x;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      x[r] = *(DEERS_LDS const float*)(uintptr_t)(lds + ds_at + (8 * (r >> 2) + (r & 3)) * 16);
    accumulate<D>(acc[0], lds, x, lane);
    settle_lds_reads();
  }
  const int qrow = 32 * qb + q;
  float* const row = (float*)p.dq + b * p.sdq.b + h * p.sdq.h + (int64_t)min(qrow, T - 1) * p.sdq.t;
  const float mul = p.scale;
  leave_sums<D, W, 1, S::WAVE>(acc, lds, lane);
  store_sums<D, W, 1, S::WAVE>(acc, lds_address(smem), nullptr, &mul, &row, qrow < T, wave, lane);
}

template <int D, int W>
void launch_bwd(const BwdParams& p, int BH, int heads, char* ds, hipStream_t stream) {
  const auto dkdv = attn_bwd_f32_dkdv_kernel<D, W>;
  const auto dq = attn_bwd_f32_dq_kernel<D, W>;
  constexpr size_t lds_dkdv = split32_lds<D, W>(), lds_dq = DqPass<D, W>::LDS;
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) allow_lds(dkdv, lds_dkdv), allow_lds(dq, lds_dq);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  for (int bh = 0; bh < BH; bh += heads) {
    const int n = std::min(heads, BH - bh);
    const dim3 grid(map_even_blocks(n_blocks, n));
    {
      LaunchScope scope("attn_bwd_dkdv", stream);
      hipLaunchKernelGGL(dkdv, grid, dim3(64 * W), lds_dkdv, stream, p, bh, n, n_blocks, ds);
    }
    LaunchScope scope("attn_bwd_dq", stream);
    hipLaunchKernelGGL(dq, grid, dim3(64 * W), lds_dq, stream, p, bh, n, n_blocks, ds);
  }
}

}  // namespace

bool attn_f32_one_wave(int64_t n, int64_t nb, int64_t D);  // attn_split_f32.hip

namespace {

// Waves per workgroup of both passes, for n workgroups that walk up to nb blocks.  As in
// attn_split_f32.hip: one where many workgroups of short walks cover the SIMDs (400 x 512 x 64: 412 us in
// four waves, 374 in two, 353 in one), four where the longest walk would be alone at the end (24 x 4096 x 64
// 1058 / 1085 / 1206), two between (192 x 384 x 64 129 / 118 / 127; 48 x 512 x 128 138 / 124 / 199).
int bwd_waves(int64_t n, int64_t nb, int64_t D) {
  if (attn_f32_one_wave(n, nb, D)) return 1;
  return n >= (D == 32 ? 1792 + 24 * nb : D == 64 ? 384 + 72 * nb : 256 + 24 * nb) ? 2 : 4;
}

template <int D>
void launch_bwd(const BwdParams& p, int BH, int heads, char* ds, hipStream_t stream) {
  const int64_t rows = (int64_t)BH * p.t_pad, nb = (p.T + 31) / 32;
  {
    LaunchScope scope("attn_bwd_prep", stream);
    hipLaunchKernelGGL(attn_bwd_prep_f32_kernel<D>, dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0,
                       stream, p, rows);
  }
  switch (bwd_waves(std::min(heads, BH) * nb, nb, D)) {
    case 1: launch_bwd<D, 1>(p, BH, heads, ds, stream); break;
    case 2: launch_bwd<D, 2>(p, BH, heads, ds, stream); break;
    case 4: launch_bwd<D, 4>(p, BH, heads, ds, stream); break;
  }
}

int64_t ds_bytes(int64_t T) {
  const int64_t nb = (T + 31) / 32;
  return nb * (nb + 1) / 2 * kDsBlock;
}

}  // namespace

// dS of as many heads as the limit holds (by default a head of 34 K rows) is in memory at a time.  Larger is
// better until a share of the heads fills the device many times over: every share has an end at which CUs are
// idle (128 MB, which the memory-side cache would hold, instead of 1 GB: 96 x 1024 x 64 316 -> 336 us, 24 x 4096 x
// 64 1065 -> 1857).
int64_t attn_bwd_f32_default_ds_limit() { return (int64_t)2304 << 20; }

// Which launches come here (the others: attn_split_f32.hip, S and dP twice but one launch).  Three
// launches and a workspace pay from enough workgroups on to fill the device, n = heads * T / 32 (D = 64: at
// 512 of them, 8 x 2048, 132 us against 157; at 384, 12 x 1024, 69 against 67).  The shorter the walks, the
// more the launches weigh: below twelve blocks several times as many workgroups (192 x 256 x 64 69 against
// 71, 96 x 256 x 64 47 against 42), below eight only with one wave per workgroup (800 x 128 x 64: 81 against
// 91; 4000 x 64 x 128: 347 against 460).
static bool takes(int64_t BH, int64_t T, int64_t D) {
  const int64_t nb = (T + 31) / 32, n = BH * nb;
  if (nb >= 12) return n >= (D == 32 ? 640 : D == 64 ? 512 : 384);
  if (nb >= 8) return n >= (D == 128 ? 640 : 1536);
  return nb >= 2 && attn_f32_one_wave(n, nb, D);
}
// Returns how many heads at a time: all of them, or an even share of those whose dS the limit holds; 0: the
// launch goes elsewhere, for a share that cannot fill the device too.
int attn_bwd_f32_heads(int64_t BH, int64_t T, int64_t D, int64_t limit) {
  const int64_t most = std::min(BH, limit / ds_bytes(T));
  if (most == 0) return 0;
  const int64_t shares = (BH + most - 1) / most, heads = (BH + shares - 1) / shares;
  return takes(heads, T, D) ? (int)heads : 0;
}
size_t attn_bwd_f32_ds_bytes(int heads, int64_t T) { return (size_t)(heads * ds_bytes(T)); }

void launch_attn_bwd_f32(const BwdParams& p, int B, int D, int heads, void* ds, hipStream_t stream) {
  switch (D) {
    case 32: launch_bwd<32>(p, B * p.H, heads, (char*)ds, stream); break;
    case 64: launch_bwd<64>(p, B * p.H, heads, (char*)ds, stream); break;
    case 128: launch_bwd<128>(p, B * p.H, heads, (char*)ds, stream); break;
  }
}

}  // namespace deers
