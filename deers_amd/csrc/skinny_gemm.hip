// y[M, N] (+)= x[M, K] @ W[K, N] for M <= 32 rows, f16 storage, f32 accumulation: the
// projections of a generation step, where the batch is the only row dimension and the
// product is a single pass over the weights (src/nn.rs:183-190 with x of 32 rows;
// 1-5 MB of weights against 50-200 KB of activations).  A library GEMM spends 7-12 us on
// such a product; this kernel is one streaming read of W.
//
// Decomposition
//   grid   one workgroup per 32 columns of W; its 4 waves split K into quarters and
//          reduce their partial sums through LDS at the end (fixed order).
//   MFMA   C^T[n, m] += W^T[n, k] x^T[k, m] on v_mfma_f32_32x32x16_f16: the lane owns
//          one row m of y; W^T fragments come from the row-major W tile in LDS through
//          ds_read_b64_tr_b16 (the same transposed read the attention kernels use for V).
//   loads  global -> LDS without registers (global_load_lds_dwordx4), 4 k-steps of 16 per
//          chunk, a ring of 3 chunks per wave (2 in flight while one is consumed).  Each
//          wave reads only the LDS it filled itself: no barrier inside the loop.
//   split  when the column blocks alone are too few to occupy the chip (N = 768 gives 24),
//          K is also split over S workgroups per column block.  All S of a block run on
//          one XCD (block id % 8), write their partial tiles to a workspace in that XCD's
//          L2, and the one that arrives last (a counter per column block, reset by that
//          workgroup) adds the S partials in index order: one launch, same bits whoever
//          is last.
//   x      optionally transformed on the way in, so that a generation step needs no launch
//          of its own for them: kSkinnyReluSq squares the positive part of every x element
//          as it leaves LDS (the MLP's activation, src/models/gpt.rs:196-203; the same
//          f32 arithmetic and single rounding as the stand-alone kernel); kSkinnyRmsNorm
//          multiplies row m of the result by (mean(x[m,:]^2) + eps)^-1/2, which is
//          rms_norm(x) @ W (src/nn.rs:244-251) without the rounding of the normalised row
//          to f16 in between; the sums of squares are taken from the x tiles the MFMAs
//          read anyway.  The latter needs a workgroup to see all of K (no split).
//   W      row-major [K][N], or packed as [N/32 column blocks][K][32]: a workgroup's share of
//          a row-major W is 64 bytes out of every row, and fetched from HBM (a generation
//          step cycles through more weights and cache than the last-level cache holds) such
//          scattered pieces cost 2-3 us per launch more than the same bytes in one run.
// A product of this size is a chain of latencies: its arguments, the first chunk, the waves' sums, the meeting.  us with
// arguments from memory, divisions by S and sums by single dwords through LDS, and as it is (32 rows, packed): 768 x 2304
// 4.19 -> 3.79, 768 x 768 3.94 -> 3.36, 3072 x 768 5.91 -> 5.67, 1024 x 256 4.82 -> 4.08.
// Shapes: K a multiple of 256 (every wave then owns whole chunks), N a multiple of 8,
// rows 16-byte aligned; the caller falls back to the library otherwise.
#include "common.h"

namespace deers {

namespace {

constexpr int kSkinnyPlain = 0, kSkinnyRmsNorm = 1, kSkinnyReluSq = 2;  // the entry point's codes
constexpr int kSkWaves = 4;
constexpr int kSkStepsPerChunk = 4;           // k-steps of 16
constexpr int kSkRing = 3;                    // chunks per wave in LDS
constexpr int kSkStepBytes = 2048;            // W tile [16 k x 32 n] + x tile [32 m x 16 k], f16
constexpr int kSkChunkBytes = kSkStepsPerChunk * kSkStepBytes;
constexpr int kSkWaveBytes = kSkRing * kSkChunkBytes;
constexpr int kSkLds = kSkWaves * kSkWaveBytes;  // 96 KB
constexpr int kSkGather = 4;                     // splits whose partials the last arrival has in flight
constexpr int kSkPieceBytes = 256 * 64;          // prefetch unit: 256 rows of a packed tile

// The first 56 bytes of the arguments are in scalar registers when a wave starts (-amdgpu-kernarg-preload-count): what the
// first requests need is among them.  `form`: M, S << 8, packed << 16.  k_per_wave is a
// multiple of 64.
template <bool ACCUMULATE, int PROLOGUE>
__global__ __launch_bounds__(256) void skinny_gemm_f16_kernel(const half_t* __restrict__ x, const half_t* __restrict__ W,
                                                              half_t* __restrict__ y, int64_t ldy, int ldx, int ldw,
                                                              int N, int k_per_wave, int form, int main_blocks,
                                                              float* __restrict__ partial, int* __restrict__ counters,
                                                              float eps, int next_tiles, int next_tile_bytes,
                                                              const char* __restrict__ next_w) {
  const int M = form & 255, S = (form >> 8) & 255, K = k_per_wave * (S * kSkWaves);
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  if ((int)blockIdx.x >= main_blocks) {
    // Prefetch role (workgroups past the product's own, on CUs the product leaves idle):
    // touch the packed weight of the product that follows, each tile from the XCD whose L2
    // its consumer will read it through (block id % 8, the same mapping as below), so that
    // product finds its weights in L2 instead of HBM.  Results are discarded.
    // A tile of K rows (64 bytes each) is cut into pieces of 256 rows, one workgroup each,
    // so that a long K does not make the prefetch outlast the product it rides on.
    const int pid = (int)blockIdx.x - main_blocks;  // main_blocks is a multiple of 8
    const int pieces = next_tile_bytes / kSkPieceBytes;
    const int q = pid >> 3;
    const int tile = (q / pieces) * 8 + (pid & 7), piece = q % pieces;
    if (tile < next_tiles) {
      // the same register-free loads as the product's own, all in flight at once; they land
      // in this wave's LDS ring, where nobody reads them
      const int pw = __builtin_amdgcn_readfirstlane(tid >> 6);
      const int per_wave = kSkPieceBytes / kSkWaves;  // 4 KB
      const char* src = next_w + (int64_t)tile * next_tile_bytes + (int64_t)piece * kSkPieceBytes +
                        (int64_t)pw * per_wave;
      const uint32_t dst = lds_address(smem) + pw * kSkWaveBytes;
      for (int i = 0; i < per_wave / 1024; ++i)
        async_load16_to_lds((const half_t*)(src + i * 1024), (uint32_t)(lane * 16),
                            dst + (uint32_t)((i % (kSkWaveBytes / 1024)) * 1024));
      wait_vmcnt<0>();  // the LDS allocation must outlive the writes into it
    }
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  // block id -> (column block, K split): the S splits of a column block share id % 8
  const int n_col_blocks = (N + 31) / 32;
  const int xcd = blockIdx.x & 7, t_id = blockIdx.x >> 3;
  // t_id / S, exact: S > 1 only with fewer than 96 column blocks, far from where the rounding could reach 0.5 / S
  const int group = __builtin_amdgcn_readfirstlane((int)(((float)t_id + 0.5f) * __builtin_amdgcn_rcpf((float)S)));  
  const int split = t_id - group * S;
  const int col_block = group * 8 + xcd;
  if (col_block >= n_col_blocks) return;
  const int n0 = col_block * 32;
  const int n_chunks = k_per_wave / (16 * kSkStepsPerChunk);
  const int k_begin = (split * kSkWaves + wave) * k_per_wave;
  const uint32_t lds_wave = lds_address(smem) + wave * kSkWaveBytes;

  // W tile of a step: lane -> row lane/4 of 16, 16-byte piece lane%4 of the 64-byte row;
  // pieces past column N repeat the last valid one (their results are never stored)
  const int w_row = lane >> 2;
  const int w_piece = min(lane & 3, (N - n0) / 8 - 1);
  const uint32_t w_lane_off = (uint32_t)((w_row * ldw + 8 * w_piece) * 2);
  // x part of a chunk [32 m][64 k]: 8 rows of 128 bytes per load (clamped to row M-1), so that a
  // load touches 8 cache lines.  Row r's 16-byte piece c sits at position c ^ (r % 8): the
  // fragment reads below take one piece of 32 rows at a time and would otherwise share banks.
  uint32_t x_lane_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    x_lane_off[i] = (uint32_t)((min(8 * i + (lane >> 3), M - 1) * ldx + 8 * ((lane & 7) ^ (lane >> 3))) * 2);
  // row-major W: the block's 32 columns start 32 elements after the previous block's, rows
  // ldw apart; packed W ([column block][K][32]): blocks K*32 apart, rows 32 apart
  const half_t* w_base = W + (int64_t)col_block * (form >> 16 ? K * 32 : 32);

  auto issue = [&](int chunk) {
    const uint32_t dst = lds_wave + (chunk % kSkRing) * kSkChunkBytes;
#pragma unroll
    for (int i = 0; i < kSkStepsPerChunk; ++i) {
      const int k0 = k_begin + (chunk * kSkStepsPerChunk + i) * 16;
      async_load16_to_lds(w_base + (int64_t)k0 * ldw, w_lane_off, dst, i * 1024);
      async_load16_to_lds(x + k_begin + chunk * 64, x_lane_off[i], dst, 4096 + i * 1024);
    }
  };
  // the addend of the columns this lane will hold at the end: requested first, so that its trip
  // to memory is over by then
  const int rp = wave & 1;  // waves 0 and 1 sum and store output columns n0 + 16 rp .. + 15
  const int c_lo = n0 + 16 * rp + 4 * g, c_hi = c_lo + 8;
  half4 old_lo = {0, 0, 0, 0}, old_hi = {0, 0, 0, 0};
  if constexpr (ACCUMULATE) {
    if (wave < 2 && (lane & 31) < M) {
      if (c_lo < N) old_lo = *(const half4*)(y + (int64_t)(lane & 31) * ldy + c_lo);
      if (c_hi < N) old_hi = *(const half4*)(y + (int64_t)(lane & 31) * ldy + c_hi);
    }
  }
  issue(0);
  if (n_chunks > 1) issue(1);

  floatx16 acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  float sum_sq = 0.f;  // kSkinnyRmsNorm: this lane's share of sum(x[m,:]^2), m = lane % 32
  for (int c = 0; c < n_chunks; ++c) {
    if (c + 2 < n_chunks) {
      issue(c + 2);
      wait_vmcnt<4 * kSkStepsPerChunk>();  // two younger chunks may still be in flight
    } else if (c + 1 < n_chunks) {
      wait_vmcnt<2 * kSkStepsPerChunk>();
    } else {
      wait_vmcnt<0>();
    }
    const char* chunk = smem + wave * kSkWaveBytes + (c % kSkRing) * kSkChunkBytes;
#pragma unroll
    for (int i = 0; i < kSkStepsPerChunk; ++i) {
      // k of slot e of lane half g in step i: 16 i + 8 g + e
      const half_t* wt = (const half_t*)chunk + (16 * i + 8 * g + ((lane & 15) >> 2)) * 32 + 4 * (lane & 3) +
                         ((lane >> 4) & 1) * 16;
      const half4 a_lo = lds_read_tr16(wt), a_hi = lds_read_tr16(wt + 4 * 32);
      const half8 a = __builtin_shufflevector(a_lo, a_hi, 0, 1, 2, 3, 4, 5, 6, 7);
      half8 b = *(const half8*)(chunk + 4096 + (lane & 31) * 128 + (((2 * i + g) ^ (lane & 7)) * 16));
      if constexpr (PROLOGUE == kSkinnyReluSq) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float r = fmaxf((float)b[e], 0.f);
          b[e] = (half_t)(r * r);
        }
      }
      if constexpr (PROLOGUE == kSkinnyRmsNorm) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum_sq = fmaf((float)b[e], (float)b[e], sum_sq);
      }
      acc = mfma_f16(a, b, acc);
    }
    // the ring slot this chunk sat in is refilled two iterations from now by this same
    // wave, after these reads have returned (the MFMAs above consumed them)
  }

  // ---- reduce the four waves' partial sums (fixed order) and write 16 bytes per lane ----
  __syncthreads();  // every wave is done with its ring: reuse the start of LDS
  float* red = (float*)smem;  // [wave][reg / 4][lane][reg % 4]
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *(floatx4*)(red + ((wave * 4 + q) * 64 + lane) * 4) = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  float* red_sq = red + kSkWaves * 16 * 64;  // [wave][lane]
  if constexpr (PROLOGUE == kSkinnyRmsNorm) red_sq[wave * 64 + lane] = sum_sq;
  __syncthreads();
  float s[8];
  if (wave < 2) {
    floatx4 t[kSkWaves][2];
#pragma unroll
    for (int w = 0; w < kSkWaves; ++w)
#pragma unroll
      for (int q = 0; q < 2; ++q) t[w][q] = *(const floatx4*)(red + ((w * 4 + 2 * rp + q) * 64 + lane) * 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] = t[0][e / 4][e % 4];
#pragma unroll
      for (int w = 1; w < kSkWaves; ++w) s[e] += t[w][e / 4][e % 4];
    }
    if constexpr (PROLOGUE == kSkinnyRmsNorm) {
      // row m's sum of squares: both lane halves of all four waves, in a fixed order
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < kSkWaves; ++w) t += red_sq[w * 64 + (lane & 31)] + red_sq[w * 64 + 32 + (lane & 31)];
      const float inv = 1.0f / sqrtf(t / (float)K + eps);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] *= inv;
    }
  }
  if (S > 1) {
    // a partial tile: [column block][split][rp][pair of sums][lane], so that a wave's accesses are
    // 512-byte runs
    typedef unsigned long long u64;
    u64* tiles = (u64*)partial + ((int64_t)col_block * S * 2 + rp) * 4 * 64 + lane;
    if (wave < 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        tiles[(split * 8 + e) * 64] = __builtin_bit_cast(u64, floatx2{s[2 * e], s[2 * e + 1]});
    }
    // The S workgroups of a column block share one XCD and so one L2: a completed store
    // (vmcnt 0) is in that L2, and relaxed device-scope atomics, which bypass the CU's
    // own cache, are all the ordering needed; no cache write-back or invalidation.
    wait_all_vmem();
    __syncthreads();
    __shared__ int last_flag;
    if (tid == 0) {
      const int arrived =
          __hip_atomic_fetch_add(counters + col_block, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_flag = arrived == S - 1;
      if (last_flag)  // ready for the next launch
        __hip_atomic_store(counters + col_block, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last_flag) return;
    if (wave < 2) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] = 0.f;
      for (int sp = 0; sp < S; sp += kSkGather) {  // index order, whoever arrived last
        u64 t[kSkGather][4];  // requested together: one trip to L2, not one per split
#pragma unroll
        for (int i = 0; i < kSkGather; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            t[i][e] = __hip_atomic_load(tiles + (min(sp + i, S - 1) * 8 + e) * 64, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < kSkGather; ++i)
          if (sp + i < S)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const floatx2 f = __builtin_bit_cast(floatx2, t[i][e]);
              s[2 * e] += f[0];
              s[2 * e + 1] += f[1];
            }
      }
    }
  }
  if (wave < 2) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const int m = lane & 31;
    const int col = n0 + 16 * rp + 8 * g;  // this lane's 8 output columns after the exchange
    // Before the exchange the lane holds columns 16rp + 4g + {0..3} (s[0..3]) and
    // 16rp + 8 + 4g + {0..3} (s[4..7]) of row m; its partner (lane ^ 32) the other halves.
    half4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = (half_t)s[e];
      hi[e] = (half_t)s[4 + e];
    }
    if constexpr (ACCUMULATE) {  // in f32, before the one rounding
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = (half_t)(s[e] + (float)old_lo[e]);
        hi[e] = (half_t)(s[4 + e] + (float)old_hi[e]);
      }
    }
    const u32x2 xu = __builtin_bit_cast(u32x2, lo), yu = __builtin_bit_cast(u32x2, hi);
    const auto r0 = __builtin_amdgcn_permlane32_swap(xu[0], yu[0], false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(xu[1], yu[1], false, false);
    if (m < M && col < N) *(u32x4*)(y + (int64_t)m * ldy + col) = u32x4{r0[0], r1[0], r0[1], r1[1]};
  }
}

}  // namespace

// true if the kernel takes this product (see the shape rules above)
bool skinny_gemm_takes(int64_t m, int64_t n, int64_t k, int64_t ldx, int64_t ldw, int64_t ldy,
                       const void* x, const void* w, const void* y) {
  if (m < 1 || m > 32 || n < 8 || n % 8 || k < 256 || k % 256) return false;
  if (ldx % 8 || ldw % 8 || ldy % 8 || ldx < k || ldw < n || ldy < n) return false;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) return false;
  if (k * ldw * 2 >= ((int64_t)1 << 31) || 32 * ldx * 2 >= ((int64_t)1 << 31)) return false;
  return true;
}

// Number of K splits per column block for this shape.  A split costs a trip through the workspace and
// the arrival counter, 0.5 to 0.9 us (1024 x 1024: 4.17 us unsplit, 4.91 in two; 768 x 768 3.81, 4.53 in three;
// 1280 x 1280 4.80, 5.79 in five), and saves the time in which a workgroup streams what it gives away.  That
// pays from K = 1536 on with shares of 512 or more (packed weights, one row; 32 rows alike): 1536 x 768 5.00 us
// unsplit, 5.19 in two, 4.97 in three; 2048 x 512 5.65, 5.34 in two, 4.93 in four; 2560 x 640 6.66, 6.01 in two, 5.51 in
// five; 3072 x 768 7.45, 5.80 in three, 5.55 in four, 5.95 in six; 4096 x 1024 8.91, 6.35 in four, 7.22 in eight.
// With 48 column blocks or more the device streams fast enough up to K = 2048 (1536 x 1536 5.21 unsplit, 5.61 in
// two; 1536 x 2304 5.22, 5.85; 2048 x 2048 5.98, 6.20; but 3072 x 2304 7.67, 7.11), and with 96 at any.
int skinny_gemm_splits(int64_t n, int64_t k) {
  const int64_t col_blocks = (n + 31) / 32, units = k / 256;  // a split owns whole 256-deep units
  if (units < 6 || col_blocks >= (units <= 8 ? 48 : 96)) return 1;
  int best = 1;
  for (int sp = 2; sp <= units / 2 && sp <= 16; ++sp)
    if (units % sp == 0) {
      best = sp;
      if (col_blocks * sp >= 96) break;
    }
  return best;
}
size_t skinny_gemm_workspace_bytes(int64_t n, int splits) {
  return splits > 1 ? (size_t)((n + 31) / 32) * splits * 2 * 64 * 8 * sizeof(float) : 0;
}

template <bool ACCUMULATE, int PROLOGUE>
static void launch_one(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy, int m,
                       int n, int k, int splits, float* partial, int* counters, float eps, bool packed,
                       const SkinnyPrefetch& next, hipStream_t stream) {
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)skinny_gemm_f16_kernel<ACCUMULATE, PROLOGUE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, kSkLds);
    attr_set = true;
  }
  const int col_blocks = (n + 31) / 32;
  const int main_blocks = 8 * splits * ((col_blocks + 7) / 8);
  const int next_tiles = next.w ? (int)((next.n + 31) / 32) : 0;
  const int pieces = next.w ? (int)(next.k / 256) : 0;  // K % 256 == 0 for every weight the kernel takes
  const dim3 grid((unsigned)(main_blocks + 8 * ((next_tiles + 7) / 8) * pieces));
  hipLaunchKernelGGL((skinny_gemm_f16_kernel<ACCUMULATE, PROLOGUE>), grid, dim3(256), kSkLds, stream,
                     (const half_t*)x, (const half_t*)w, (half_t*)y, ldy, (int)ldx, packed ? 32 : (int)ldw, n, k / (splits * kSkWaves),
                     m | splits << 8 | (int)packed << 16, main_blocks, partial, counters, eps, next_tiles,
                     (int)(next.k * 64), (const char*)next.w);
}

// prologue: kSkinnyPlain, kSkinnyRmsNorm (splits must be 1) or kSkinnyReluSq; packed: w is
// [ceil(n/32)][k][32] (each workgroup's columns contiguous) instead of row-major
void launch_skinny_gemm_f16(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy,
                            int m, int n, int k, bool accumulate, int prologue, float eps, bool packed,
                            int splits, float* partial, int* counters, const SkinnyPrefetch& next,
                            hipStream_t stream) {
#define DEERS_SKINNY_CASE(ACC, PRO)                                                                      \
  if (accumulate == ACC && prologue == PRO)                                                              \
    return launch_one<ACC, PRO>(x, ldx, w, ldw, y, ldy, m, n, k, splits, partial, counters, eps, packed, next, stream);
  DEERS_SKINNY_CASE(false, kSkinnyPlain)
  DEERS_SKINNY_CASE(true, kSkinnyPlain)
  DEERS_SKINNY_CASE(false, kSkinnyRmsNorm)
  DEERS_SKINNY_CASE(true, kSkinnyRmsNorm)
  DEERS_SKINNY_CASE(false, kSkinnyReluSq)
  DEERS_SKINNY_CASE(true, kSkinnyReluSq)
#undef DEERS_SKINNY_CASE
}

}  // namespace deers
