// Fused causal attention for launches that cannot fill the device, f16 storage / f32
// accumulate, gfx950: forward and backward of the same contract as attn_fwd_f16.hip and
// attn_bwd_f16.hip (src/models/gpt.rs:139-144; src/ops.rs:1089-1101, 422-425, 210-214, 777-799,
// 1162-1175, 638-643).
//
// The kernels of those files give a workgroup 128 rows and let its four waves walk the other
// operand together: one dependent chain of T / 32 stages with a barrier in each.  With few heads
// or short sequences the launch is nothing but that chain (12 heads of 512 x 64: 48 workgroups on
// 256 CUs, forward 10.1 us and backward 17.5 us; here 5.5 and 8.0).  Here a workgroup owns 32 rows,
// so there are four times as many of them, and its W waves divide the blocks of 32 rows of the
// other operand among themselves (wave w takes blocks w, w + W, ...), each with its own loads,
// its own slice of LDS and no barrier; their partial results meet once, at the end, in LDS.  The
// chain of a wave is T / (32 W) stages.  The price is that nothing is shared between waves: every
// 32 rows read all of the other operand through L1 (64 bytes per clock and CU), so launches that
// fill the device anyway stay with the 128-row kernels (the rule is above split_takes, below).
//
//   forward  S^T = K Q^T, one query per lane; online softmax per wave; O, m and l are merged.
//   dQ       the same walk: S^T and dP^T = V dO^T, dQ^T += K^T dS^T; sums merged.
//   dK/dV    a workgroup owns 32 keys, one per lane, and walks Q and dO.  It forms each query block's row sums
//            dO . O itself, so it waits for nobody: no workspace, no flags, nothing to hand over between workgroups.
// The walked operands pass through LDS, rows and transposed fragments from the same blocks; what a workgroup owns is
// loaded once through LDS as well, by all its waves.  All three form the scores from Q and apply scale * log2e to the
// f32 sums; where the 128-row backward follows the forward (or, in a captured launch, the 128-row forward has gone
// before), from what that takes, Q or f16(Q * scale * log2e): a probability is recomputed from the score it was
// normalised with (attn_f16_from_q).  Partial sums are added in wave order: results are reproducible bit for bit.
//
// What bounds a launch: the start of a workgroup (2 us of loads that depend on nothing but its number), the stages of
// its longest wave (1.0 us at D = 128 and 0.6 us at D = 64 in the backward, for 0.5 and 0.25 us of matrix
// instructions: fragments from LDS, 1 KB per instruction, and what cannot be issued behind one), and the merge with
// its stores (1.5 us); with the device full, LDS reads.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace deers {

namespace {

using rsrc_t = __amdgpu_buffer_rsrc_t;

// A 32-row block in LDS is filled by loads of 1 KB, 64 lanes of 16 bytes, and read in two ways without bank conflicts:
// 16 bytes of 16 rows, and 8 bytes of 4 rows x 4 chunks of 16 bytes.  A lane of a load takes one chunk of one row:
//   D = 128  the load's 4 rows by groups of 4 chunks, [chunk / 4][row][chunk % 4], the next load 16 bytes further on:
//            every fragment's address is the lane's part plus a constant;
//   else     row after row, chunk c at position c ^ lds_swizzle(row).  (The constant form would have neighbouring
//            lanes read 32 bytes of a row instead of 64 and more.)
template <int D>
struct SplitCfg {
  static constexpr int KS = D / 16;         // contraction steps over D
  static constexpr int DB = D / 32;         // 32-wide blocks of D
  static constexpr int RB = 2 * D;          // bytes per row
  static constexpr int CH = D / 8;          // 16-byte chunks per row
  static constexpr int NI = 32 * RB / 1024;  // loads per block
  static constexpr int RPL = 32 / NI;        // rows per load
  static constexpr int LB = D == 128 ? 1024 + 16 : 1024;  // from load to load in LDS
  static constexpr int BB = NI * LB;         // bytes of a block
  static __device__ __forceinline__ int load_row(int i, int lane) {
    return i * RPL + (D == 128 ? (lane >> 2) & 3 : lane / CH);
  }
  static __device__ __forceinline__ int load_chunk(int i, int lane) {
    return D == 128 ? (lane & 3) + 4 * (lane >> 4) : (lane % CH) ^ lds_swizzle<CH>(load_row(i, lane));
  }
};

// Every load of this wave has landed, those into LDS included; LDS reads stay behind it.
__device__ __forceinline__ void settle_loads() {
  wait_all_vmem();
  asm volatile("" ::: "memory");
}

// Requests rows r0 .. r0 + 31 (rows past T - 1 read row T - 1) of a [T, D] matrix into the block at LDS address `dst`.
template <int D>
__device__ __forceinline__ void split_load_block(const half_t* base, int row_stride, int r0, int T, uint32_t dst,
                                                 int lane) {
  using C = SplitCfg<D>;
#pragma unroll
  for (int i = 0; i < C::NI; ++i)
    async_load16_to_lds(base, (uint32_t)min(r0 + C::load_row(i, lane), T - 1) * (uint32_t)row_stride * 2 +
                                  16 * C::load_chunk(i, lane), dst, i * C::LB);
}

template <int N, int I = 0, typename F>
__device__ __forceinline__ void split_for(F&& f) {  // f(0), .., f(N - 1) as compile-time constants
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    split_for<N, I + 1>(f);
  }
}

// The 32-row blocks of one head of a [B,H,T,D] tensor on their way into LDS, through a descriptor that ends with the
// head's last row: rows past it become zeros, and so does a whole block past the end, which a wave asks for that
// has none left, so that a stage has no branch around its requests.  The lane's part of an address is kept in
// registers (T < 32: not used, rows of one block may be further apart than an offset reaches), a block's is one
// scalar.
template <int D>
struct SplitStream {
  using C = SplitCfg<D>;
  static constexpr int NOFF = D == 128 ? 1 : C::NI;  // D = 128: load after load 4 rows on, the same chunks
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  static constexpr uint32_t kShift = 2048;  // the descriptor starts that many bytes before the head
  u32x4 rsrc;
  uint32_t stride;  // bytes
  uint32_t off[NOFF];

  __device__ __forceinline__ SplitStream(const void* tensor, const Strides3& s, int b, int h, int T, int lane)
      : stride((uint32_t)s.t * 2) {
    const uint64_t at = uniform_address((const half_t*)tensor + b * s.b + h * s.h) - kShift;
    rsrc = u32x4{(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, (uint32_t)(T - 1) * stride + C::RB + kShift, 0x00020000u};
#pragma unroll
    for (int i = 0; i < NOFF; ++i) off[i] = (uint32_t)C::load_row(i, lane) * stride + 16 * C::load_chunk(i, lane);
  }
  // Loads I and I + 1 of a block to the block at LDS address `dst`, with one write of m0: an instruction's offset counts
  // in memory and in LDS, so the second load's other part is short of it (by at most LB, which kShift makes up for).
  // Wait states: one from the write of m0; five in case a vector instruction has just written one of the scalar
  // registers (readlane, where scalars were spilled).  What is left is seven issue slots, less than two matrix
  // instructions hide; all requests of a stage behind its first products took 120 clocks a pair.
  template <int I>
  __device__ __forceinline__ void request(int block, uint32_t dst) const {
    const uint32_t at = __builtin_amdgcn_readfirstlane(dst);
    const uint32_t first = 32u * (uint32_t)block * stride + kShift + (D == 128 ? I * C::RPL * stride : 0);
    const uint32_t second = first - C::LB + (D == 128 ? C::RPL * stride : 0);
    asm volatile("s_add_u32 m0, %5, %6\n\ts_nop 3\n\t"
                 "buffer_load_dwordx4 %0, %2, %3 offen lds\n\t"
                 "buffer_load_dwordx4 %1, %2, %4 offen offset:%7 lds"
                 ::"v"(off[D == 128 ? 0 : I]), "v"(off[D == 128 ? 0 : I + 1]), "s"(rsrc), "s"(first), "s"(second), "s"(at),
                   "i"(I * C::LB), "i"(C::LB)
                 : "memory", "scc");
  }
  // A whole block, for any T.
  __device__ __forceinline__ void request_all(int block, const void* tensor, const Strides3& s, int b, int h, int T,
                                              uint32_t dst, int lane) const {
    if (T >= 32)
      split_for<C::NI / 2>([&](auto i) { request<2 * decltype(i)::value>(block, dst); });
    else
      split_load_block<D>((const half_t*)tensor + b * s.b + h * s.h, (int)s.t, 32 * block, T, dst, lane);
  }
};

// Rows r0 .. r0 + 31 (past T - 1: row T - 1) of N = 1 or 2 matrices, which all waves of a workgroup hold in registers,
// into adjoining blocks at LDS address `dst`, each wave its share: whole cache lines, once per workgroup.
template <int D, int W, int N = 2>
__device__ __forceinline__ void split_load_resident(const void* x, const Strides3& sx, const void* y, const Strides3& sy, int b,
                                                    int h, int r0, int T, uint32_t dst, int wave, int lane) {
  using C = SplitCfg<D>;
  constexpr int per = (N * C::NI + W - 1) / W;
  const half_t* const bx = (const half_t*)x + b * sx.b + h * sx.h;
  const half_t* const by = (const half_t*)y + b * sy.b + h * sy.h;
#pragma unroll
  for (int j = 0; j < per; ++j) {
    const int load = wave * per + j, i = load % C::NI;
    if (N * C::NI % W && load >= N * C::NI) break;
    const uint32_t stride = (uint32_t)(load < C::NI ? sx.t : sy.t) * 2;
    async_load16_to_lds(load < C::NI ? bx : by,
                        (uint32_t)min(r0 + C::load_row(i, lane), T - 1) * stride + 16 * C::load_chunk(i, lane), dst,
                        load * C::LB);
  }
}

// Row sums dO . O of a block whose dO is in LDS.
//   D = 32   from the fragments of dO's rows and O in the same layout, 16 bytes of 32 rows per load: two loads.
//   else     such loads occupy the address unit eight times as long as whole cache lines do.  A lane takes the chunks
//            of O that it would load into LDS, and the same chunks of dO; what the lanes of a row have is summed
//            through LDS.
//   D = 128  A load's lanes are, 16 by 16, 4 rows x 4 chunks, the next 16 the rows' next chunks, which is what a
//            16 x 16 x 32 product contracts: its diagonal holds the sums over every fourth chunk (16 clocks of the
//            matrix unit; v_dot2 takes 16 for two elements of a lane's eight).
template <int D>
struct SplitRowDots {
  using C = SplitCfg<D>;
  static constexpr int LD = C::CH + 4;  // floats from row to row: reads of a quarter of the rows on all banks
  static constexpr int kFloats = D == 32 ? 0 : 32 * LD;
  static constexpr int NOFF = D == 64 ? C::NI : 1;
  typedef std::conditional_t<D == 128, floatx4, float> Part;
  uint32_t off[NOFF];
  uint32_t stride;

  __device__ __forceinline__ SplitRowDots(const Strides3& s, int T, int lane) : stride((uint32_t)s.t * 2) {
    if constexpr (D == 32) {
      off[0] = (uint32_t)min(lane & 31, T - 1) * stride + 16 * (lane >> 5);
    } else {
#pragma unroll
      for (int i = 0; i < NOFF; ++i)
        off[i] = (uint32_t)min(C::load_row(i, lane), T - 1) * stride + 16 * C::load_chunk(i, lane);
    }
  }
  // O's descriptor; reads past the last row give zeros
  static __device__ __forceinline__ rsrc_t rsrc(const void* tensor, const Strides3& s, int b, int h, int T) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)((const half_t*)tensor + b * s.b + h * s.h), 0,
                                             (int)((uint32_t)(T - 1) * (uint32_t)s.t * 2 + C::RB), 0x00020000);
  }
  __device__ __forceinline__ half8 load(rsrc_t r, int i, int block) const {
    const uint32_t first = 32u * (uint32_t)block * stride + (D == 128 ? i * C::RPL * stride : 0);
    return __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off[D == 64 ? i : 0] + (D == 32 ? 32 * i : 0),
                                                                           (int)first, 0));
  }
  static __device__ __forceinline__ Part multiply(half8 o, half8 d) {
    if constexpr (D == 128) {
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(o, d, floatx4{0, 0, 0, 0}, 0, 0, 0);
    } else {
      float t = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) t = __builtin_amdgcn_fdot2(half2v{o[e], o[e + 1]}, half2v{d[e], d[e + 1]}, t, false);
      return t;
    }
  }
  static __device__ __forceinline__ void leave(float* parts, const Part (&t)[C::NI], int lane) {
    if constexpr (D == 128) {
      if (((lane >> 2) & 3) == lane >> 4) {  // lanes with a diagonal element, in register lane % 4
#pragma unroll
        for (int i = 0; i < C::NI; ++i) *(floatx4*)(parts + C::load_row(i, lane) * LD + 4 * (lane & 3)) = t[i];
      }
    } else if constexpr (D == 64) {
#pragma unroll
      for (int i = 0; i < C::NI; ++i) parts[C::load_row(i, lane) * LD + lane % C::CH] = t[i];
    }
  }
  // the sum of row lane % 32
  static __device__ __forceinline__ float sum(const float* parts, const Part (&t)[C::NI], int lane) {
    if constexpr (D == 32) {
      return pair_sum(t[0] + t[1]);
    } else if constexpr (D == 64) {
      const floatx4 x = *(const floatx4*)(parts + (lane & 31) * LD + (lane >> 5) * 4);
      return pair_sum((x[0] + x[1]) + (x[2] + x[3]));
    } else {
      const float* row = parts + (lane & 31) * LD;
      return (row[0] + row[5]) + (row[10] + row[15]);
    }
  }
};

// LDS addresses of a lane's fragments in a block, kept in registers over a walk: a stage moves them to its slot by one
// addition each, and what is constant in a read goes into its offset.
template <int D>
struct SplitFrags {
  using C = SplitCfg<D>;
  static constexpr bool kFlat = D == 128;
  static constexpr int NR = kFlat ? 1 : C::KS, NC = kFlat ? 1 : C::DB * 2;
  uint32_t row_at[NR];  // row lane % 32, halfs 16 ks + 8 g ..
  uint32_t col_at[NC];  // column 32 db + lane % 32, rows {4g .. 4g+3} and {8+4g .. 8+4g+3}
  __device__ __forceinline__ SplitFrags(uint32_t block, int lane) {
    const int r = lane & 31, g = lane >> 5, c4 = lane & 3;
    const int lrow = 4 * g + ((lane & 15) >> 2), c_lo = 2 * ((lane >> 4) & 1) + (c4 >> 1);
    if constexpr (kFlat) {
      row_at[0] = block + (r >> 2) * C::LB + (r & 3) * 64 + g * 16;
      col_at[0] = block + g * C::LB + (lrow & 3) * 64 + c_lo * 16 + (c4 & 1) * 8;
    } else {
#pragma unroll
      for (int ks = 0; ks < C::KS; ++ks)
        row_at[ks] = block + r * C::RB + (((2 * ks + g) ^ lds_swizzle<C::CH>(r)) << 4);
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int row = lrow + 8 * (n & 1);
        col_at[n] = block + row * C::RB + (((4 * (n >> 1) + c_lo) ^ lds_swizzle<C::CH>(row)) << 4) + (c4 & 1) * 8;
      }
    }
  }
  __device__ __forceinline__ void move(uint32_t by) {
#pragma unroll
    for (int n = 0; n < NR; ++n) row_at[n] = opaque(row_at[n] + by);
#pragma unroll
    for (int n = 0; n < NC; ++n) col_at[n] = opaque(col_at[n] + by);
  }
  // fragment ks of the lane's row; `offset`: another block
  __device__ __forceinline__ half8 row(int ks, uint32_t offset = 0) const {
    return kFlat ? lds_read_half8_at(row_at[0] + offset + (ks & 1) * 32 + (ks >> 1) * 256)
                 : lds_read_half8_at(row_at[kFlat ? 0 : ks] + offset);
  }
  // transposed fragment: rows 16 ms + {4g .. 4g+3, 8+4g .. 8+4g+3}, the order in which registers 8 ms .. 8 ms + 7 of
  // an accumulator hold their rows
  __device__ __forceinline__ half8 col(int ms, int db, uint32_t offset = 0) const {
    const half4 lo = lds_read_tr16_at(kFlat ? col_at[0] + offset + 4 * ms * C::LB + db * 256
                                            : col_at[kFlat ? 0 : 2 * db] + offset + 16 * ms * C::RB);
    const half4 hi = lds_read_tr16_at(kFlat ? col_at[0] + offset + (4 * ms + 2) * C::LB + db * 256
                                            : col_at[kFlat ? 0 : 2 * db + 1] + offset + 16 * ms * C::RB);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// The fragments of rows r0 + lane % 32 (past T - 1: row T - 1) of a head, straight into registers: at D = 32, two loads,
// less than the way through LDS (kSplitDirect).
template <int D>
constexpr bool kSplitDirect = D == 32;
template <int D>
__device__ __forceinline__ void split_global_frags(half8* f, const void* tensor, const Strides3& s, int b, int h, int r0, int T,
                                                   int lane) {
  const half_t* p = (const half_t*)tensor + b * s.b + h * s.h + (int64_t)min(r0 + (lane & 31), T - 1) * s.t + 8 * (lane >> 5);
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
__device__ __forceinline__ half8 pack_regs(const floatx16& a, int ms) {
  half8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (half_t)a[8 * ms + e];
  return r;
}

// Results of [32 rows, D] (row = lane % 32, register r of block db is column 32 db + 8 (r / 4) + 4 g + r % 4) meet
// by units of 16 columns, 8 registers: every wave leaves its accumulators in its own LDS, `own_lds` and on (32 rows x
// D floats per result, what the wave's blocks took), and of the units of the N results together wave w sums
// w, w + W, .. in wave order, after one barrier.  Which wave owns a unit is an address only: this code runs once per
// workgroup, and its length costs more than the reads it could save.
template <int D, int W>
struct SplitMerge {
  using C = SplitCfg<D>;
  static constexpr int U = 2 * C::DB;
  static constexpr int kUnitBytes = 8 * 64 * 4;
  static constexpr int kWaveBytes = U * kUnitBytes;  // of one result

  template <int N>
  static __device__ __forceinline__ void leave(const floatx16 (&acc)[N][C::DB], uint32_t own_lds, int lane) {
    if constexpr (W == 1) return;
#pragma unroll
    for (int q = 0; q < N * U * 2; ++q) {
      const floatx16& a = acc[q / 2 / U][q / 2 % U / 2];
      const int r = 4 * (q % 4);
      *(DEERS_LDS floatx4*)(uintptr_t)(own_lds + lane * 16 + q * 1024) = floatx4{a[r], a[r + 1], a[r + 2], a[r + 3]};
    }
    __syncthreads();
  }
  // first_lds: wave 0's, the others' WAVE_BYTES apart; weight[w]: of wave w's part.  Rows go to dst[n] (this lane's
  // row; not where !store), times mul[n].
  template <int N, bool WEIGHTED, int WAVE_BYTES>
  static __device__ __forceinline__ void gather(const floatx16 (&acc)[N][C::DB], uint32_t first_lds, const float* weight,
                                                const float* mul, half_t* const* dst, bool store, int wave, int lane) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    static_assert(WAVE_BYTES >= N * kWaveBytes);
#pragma unroll
    for (int j = 0; j < (N * U + W - 1) / W; ++j) {
      const int u = W == 1 ? j : j * W + wave;
      if (N * U % W && u >= N * U) break;
      float sum[8];
      if constexpr (W == 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = acc[j / U][j % U / 2][8 * (j % 2) + e] * (WEIGHTED ? weight[0] : 1.f);
      } else {
        const uint32_t at = first_lds + u * kUnitBytes + lane * 16;
#pragma unroll
        for (int w = 0; w < W; ++w) {
          const floatx4 t[2] = {lds_read_float4_at(at + w * WAVE_BYTES), lds_read_float4_at(at + w * WAVE_BYTES + 1024)};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = t[e / 4][e % 4];
            if (WEIGHTED)
              sum[e] = w ? fmaf(v, weight[w], sum[e]) : v * weight[0];
            else
              sum[e] = w ? sum[e] + v : v;
          }
        }
      }
      const bool second = N > 1 && u >= U;
      const float f = second ? mul[N - 1] : mul[0];
      half_t* const row = second ? dst[N - 1] : dst[0];
      half4 x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = (half_t)(sum[e] * f);
        y[e] = (half_t)(sum[4 + e] * f);
      }
      // the lane pair (l, l ^ 32) trades halves so that each stores 16 contiguous bytes
      const u32x2 xu = __builtin_bit_cast(u32x2, x), yu = __builtin_bit_cast(u32x2, y);
      const auto r0 = __builtin_amdgcn_permlane32_swap(xu[0], yu[0], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(xu[1], yu[1], false, false);
      if (store) *(u32x4*)(row + 16 * (u % U) + 8 * (lane >> 5)) = u32x4{r0[0], r1[0], r0[1], r1[1]};
    }
  }
};

// A stage is one stream of instructions: a wave is alone on its SIMD or nearly so, and what it issues behind a matrix
// instruction is free, while its own waits are not.  So the order is written down.  Forward: S, with requests for the
// next block behind its products, the softmax, P V.  Backward: S; dP, with the exponentials of S behind its products;
// then the products that consume P and dS, with the multiplications and roundings that make dS behind them.
#define DEERS_SPLIT_CHUNK_END() __builtin_amdgcn_sched_barrier(0)
constexpr int kSplitAhead = 4;  // fragments on their way from LDS: a read takes four matrix instructions

// ---- forward ----

// DOUBLE: K and V have two blocks each per wave, the next ones are requested while this one's are in use.  Otherwise
// one each, asked for again as soon as they have been read: half the LDS, for launches in which several waves of a
// SIMD cover each other's waits.
// One wave: Q passes through V's block, V is asked for after it (a third more workgroups per CU).
// DOUBLE at D = 32: K's rows go straight into registers a stage ahead (kSplitKDirect) and V is asked for when the stage
// begins: the stage is a chain of waits, and this takes the read of K from LDS off it and gives V all of it (3 heads x
// 2038 9.50 -> 8.41 us, 8 x 502 4.32 -> 4.07).
template <int D, int W, bool DOUBLE>
constexpr bool kSplitQInV = W == 1 && !DOUBLE && !kSplitDirect<D>;
template <int D, bool DOUBLE>
constexpr bool kSplitKDirect = kSplitDirect<D> && DOUBLE;
template <int D, int W, bool DOUBLE>
constexpr size_t split_fwd_lds() {  // blocks of every wave, as large as its accumulators; Q's block; m and l of every wave
  static_assert(2 * SplitCfg<D>::BB >= SplitMerge<D, W>::kWaveBytes, "the merge takes the blocks' place");
  return (size_t)(W * (DOUBLE ? 4 : 2) + (kSplitQInV<D, W, DOUBLE> || kSplitDirect<D> ? 0 : 1)) * SplitCfg<D>::BB + W * 32 * 2 * sizeof(float);
}

template <int D, int W, bool DOUBLE>
__global__ __launch_bounds__(64 * W, 2) void attn_fwd_f16_split_kernel(FwdParams p, int BH, int n_blocks, int cus,
                                                                      int scaled_q) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB, A = kSplitAhead, kWave = (DOUBLE ? 4 : 2) * C::BB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  fetch_arguments<decltype(attn_fwd_f16_split_kernel<D, W, DOUBLE>)>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, T = p.T;
  int bh, rank;
  if (!map_block_even(D == 128 ? paired_block(blockIdx.x, gridDim.x, cus) : blockIdx.x, n_blocks, BH, &bh, &rank)) return;
  const int qb = n_blocks - 1 - rank;  // longest rows first
  const int b_ = bh / p.H, h_ = bh % p.H;
  const int qrow = 32 * qb + (lane & 31);
  const uint32_t ring = lds_address(smem) + wave * kWave;
  constexpr bool kQInV = kSplitQInV<D, W, DOUBLE>;
  const uint32_t q_blk = lds_address(smem) + (kQInV ? C::BB : W * kWave);

  half8 qf[KS];
  if constexpr (kSplitDirect<D>)
    split_global_frags<D>(qf, p.q, p.sq, b_, h_, 32 * qb, T, lane);
  else
    split_load_resident<D, W, 1>(p.q, p.sq, p.q, p.sq, b_, h_, 32 * qb, T, q_blk, wave, lane);
  const SplitStream<D> K(p.k, p.sk, b_, h_, T, lane), V(p.v, p.sv, b_, h_, T, lane);
  constexpr bool kKDirect = kSplitKDirect<D, DOUBLE>;
  const SplitRowDots<D> k_rows(p.sk, T, lane);
  const rsrc_t k_rsrc = k_rows.rsrc(p.k, p.sk, b_, h_, T);
  half8 kf[KS];
  int kb = wave;
  if (kb <= qb) {
    if constexpr (kKDirect) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = k_rows.load(k_rsrc, ks, kb);
    } else {
      K.request_all(kb, p.k, p.sk, b_, h_, T, ring, lane);
    }
    if (!kQInV) V.request_all(kb, p.v, p.sv, b_, h_, T, ring + C::BB, lane);
  }
  const float c = scaled_q ? 1.f : p.scale_log2;
  floatx16 oacc[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[0][db] = ZERO16;
  settle_loads();
  if constexpr (!kSplitDirect<D>) {
    __syncthreads();
    const SplitFrags<D> at(q_blk, lane);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = at.row(ks);
  }
  if (kQInV) {
    settle_lds_reads();
    V.request_all(kb, p.v, p.sv, b_, h_, T, ring + C::BB, lane);
  }
  if (scaled_q) scale_frags<KS>(qf, p.scale_log2);

  float m = -INFINITY, l = 0.f;
  SplitFrags<D> at(ring, lane);
  uint32_t slot = 0;
  for (; kb <= qb; kb += W) {
    const bool more = kb + W <= qb;
    const int next = more ? kb + W : n_blocks;
    const uint32_t other = DOUBLE ? slot ^ (2 * C::BB) : 0;
    if constexpr (DOUBLE)
      settle_loads();  // K and V of this block
    else
      wait_vmcnt<C::NI>();  // K; V's block may be on its way
    // fragments in the order of their use: K rows, V columns
    half8 f[A];
    auto fetch = [&](auto i) {
      constexpr int n = decltype(i)::value;
      if constexpr (n < KS)
        f[n % A] = at.row(n);
      else if constexpr (n < KS + 2 * DB)
        f[n % A] = at.col((n - KS) / DB, (n - KS) % DB, C::BB);
    };
    half8 k_next[KS];
    if constexpr (kKDirect) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) k_next[ks] = k_rows.load(k_rsrc, ks, next);
      split_for<2 * DB>([&](auto i) { fetch(std::integral_constant<int, KS + decltype(i)::value>()); });
    } else {
      split_for<(DOUBLE || A < KS ? A : KS)>(fetch);
    }
    floatx16 s = ZERO16;
    DEERS_SPLIT_CHUNK_END();
    split_for<KS>([&](auto i) {
      constexpr int ks = decltype(i)::value;
      s = mfma_f16(kKDirect ? kf[ks] : f[ks % A], qf[ks], s);
      if constexpr (!kKDirect && (DOUBLE || ks + A < KS)) fetch(std::integral_constant<int, ks + A>());
      if constexpr (kKDirect && ks % 2 == 0)
        V.template request<ks>(next, ring + other + C::BB);
      else if constexpr (DOUBLE && ks % 2 == 0)
        K.template request<ks>(next, ring + other);
      DEERS_SPLIT_CHUNK_END();
    });
    if (!DOUBLE && more) {  // K's block has been read
      settle_lds_reads();
      split_for<KS / 2>([&](auto i) { K.template request<2 * decltype(i)::value>(next, ring); });
    }
    if (kb == qb) {  // the diagonal block (its keys past T - 1 lie in the future of every stored row)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
    float mx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) mx[i] = fmaxf(fmaxf(s[i], s[i + 4]), fmaxf(s[i + 8], s[i + 12]));
    const float top = pair_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]))) * c;
    const float m_new = fmaxf(m, top);
    if (__any(m_new > m)) {  // (moved later, the largest probability is no longer exact: O 2 % further off)
      const float alpha = fast_exp2(m - m_new);  // 0 in the first block
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[0][db] *= alpha;
      m = m_new;
    }
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], c, -m));
      sum[r & 1] += s[r];
    }
    l += sum[0] + sum[1];
    const half8 pf[2] = {pack_regs(s, 0), pack_regs(s, 1)};
    if constexpr (!DOUBLE) {
      if (more)
        wait_vmcnt<C::NI>();  // V; the next K is on its way
      else
        wait_vmcnt<0>();
      split_for<(A < 2 * DB ? A : 2 * DB)>([&](auto i) { fetch(std::integral_constant<int, KS + decltype(i)::value>()); });
    }
    DEERS_SPLIT_CHUNK_END();
    split_for<2 * DB>([&](auto i) {
      constexpr int n = decltype(i)::value;
      oacc[0][n % DB] = mfma_f16(f[(KS + n) % A], pf[n / DB], oacc[0][n % DB]);
      fetch(std::integral_constant<int, KS + n + A>());
      if constexpr (!kKDirect && DOUBLE && n % 2 == 0) V.template request<n>(next, ring + other + C::BB);
      DEERS_SPLIT_CHUNK_END();
    });
    if constexpr (kKDirect) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = k_next[ks];
    }
    if constexpr (DOUBLE) {
      at.move(other - slot);
      slot = other;
    } else if (more) {  // V's block has been read
      settle_lds_reads();
      split_for<KS / 2>([&](auto i) { V.template request<2 * decltype(i)::value>(next, ring + C::BB); });
    }
  }

  // ---- the waves' (m, l, O) become one; a wave without a block has m = -inf and weight 0 ----
  float* stat_m = (float*)(smem + split_fwd_lds<D, W, DOUBLE>()) - 2 * W * 32;
  float* stat_l = stat_m + W * 32;
  l = pair_sum(l);
  if (g == 0) {
    stat_m[wave * 32 + lane] = m;
    stat_l[wave * 32 + lane] = l;
  }
  if (DOUBLE) settle_loads();  // the zeros that the last stage asked for
  settle_lds_reads();
  SplitMerge<D, W>::leave(oacc, ring, lane);
  if (W == 1) __syncthreads();
  float M = -INFINITY, L = 0.f, weight[W];
#pragma unroll
  for (int w = 0; w < W; ++w) M = fmaxf(M, stat_m[w * 32 + (lane & 31)]);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    weight[w] = fast_exp2(stat_m[w * 32 + (lane & 31)] - M);
    L += stat_l[w * 32 + (lane & 31)] * weight[w];
  }
  half_t* const orow = (half_t*)p.o + b_ * p.so.b + h_ * p.so.h + (int64_t)min(qrow, T - 1) * p.so.t;
  const float inv = 1.f / L;
  SplitMerge<D, W>::template gather<1, true, kWave>(oacc, lds_address(smem), weight, &inv, &orow, qrow < T, wave, lane);
  if (wave == 0 && g == 0 && qrow < T) p.lse[(int64_t)bh * T + qrow] = (M + fast_log2(L)) * kLn2;
}

// ---- backward ----

template <int D>
constexpr int kSplitStat = 64 + SplitRowDots<D>::kFloats;  // floats per wave: row statistics, parts of the row sums
template <int D, int W>
constexpr size_t split_bwd_lds() {  // two blocks of two operands per wave, as large as its accumulators; the above
  static_assert(4 * SplitCfg<D>::BB >= 2 * SplitMerge<D, W>::kWaveBytes, "the merge takes the blocks' place");
  return (size_t)W * 4 * SplitCfg<D>::BB + W * kSplitStat<D> * sizeof(float);
}

template <int D, int W, bool SCALED_Q>
__device__ __forceinline__ void split_dq_body(const BwdParams& p, int bh, int qb, int n_blocks, char* smem, int wave,
                                              int lane) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB, A = kSplitAhead;
  const int g = lane >> 5, T = p.T;
  const int b_ = bh / p.H, h_ = bh % p.H;
  const int qrow = 32 * qb + (lane & 31), qread = min(qrow, T - 1);
  const uint32_t ring = lds_address(smem) + wave * 4 * C::BB;
  const uint32_t resident = lds_address(smem) + 2 * C::BB;  // wave 0's second slot: Q, dO
  float* stat = (float*)(smem + W * 4 * C::BB) + wave * kSplitStat<D>;

  half8 qf[KS], dof[KS];
  if constexpr (kSplitDirect<D>) {
    split_global_frags<D>(qf, p.q, p.sq, b_, h_, 32 * qb, T, lane);
    split_global_frags<D>(dof, p.d_o, p.sdo, b_, h_, 32 * qb, T, lane);
  } else {
    split_load_resident<D, W>(p.q, p.sq, p.d_o, p.sdo, b_, h_, 32 * qb, T, resident, wave, lane);
  }
  const SplitRowDots<D> dots(p.so, T, lane);
  half8 o[C::NI];
  {
    const rsrc_t r = dots.rsrc(p.o, p.so, b_, h_, T);
#pragma unroll
    for (int i = 0; i < C::NI; ++i) o[i] = dots.load(r, i, qb);
  }
  const float lse2 = -p.lse[(int64_t)bh * T + qread] * kLog2e;
  const SplitStream<D> K(p.k, p.sk, b_, h_, T, lane), V(p.v, p.sv, b_, h_, T, lane);
  int kb = wave;
  if (kb <= qb) {
    K.request_all(kb, p.k, p.sk, b_, h_, T, ring, lane);
    V.request_all(kb, p.v, p.sv, b_, h_, T, ring + C::BB, lane);
  }
  const float c = SCALED_Q ? 1.f : p.scale_log2;
  floatx16 dq[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[0][db] = ZERO16;
  settle_loads();
  if constexpr (!kSplitDirect<D>) {
    __syncthreads();
    const SplitFrags<D> at(resident, lane);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = at.row(ks);
      dof[ks] = at.row(ks, C::BB);
    }
  }
  typename SplitRowDots<D>::Part parts[C::NI];
#pragma unroll
  for (int i = 0; i < C::NI; ++i)
    parts[i] = dots.multiply(o[i], D == 32 ? dof[i] : lds_read_half8_at(resident + C::BB + i * C::LB + lane * 16));
  dots.leave(stat + 64, parts, lane);
  if (SCALED_Q) scale_frags<KS>(qf, p.scale_log2);
  const float nd = -dots.sum(stat + 64, parts, lane);
  if constexpr (!kSplitDirect<D>) {
    settle_lds_reads();
    __syncthreads();  // the second slots are free
  }

  SplitFrags<D> at(ring, lane);
  uint32_t slot = 0;
  for (; kb <= qb; kb += W) {
    settle_loads();
    const uint32_t other = slot ^ (2 * C::BB);
    const int next = kb + W <= qb ? kb + W : n_blocks;
    // fragments in the order of their use: K rows, V rows, K columns
    half8 f[A];
    auto fetch = [&](auto i) {
      constexpr int n = decltype(i)::value;
      if constexpr (n < KS)
        f[n % A] = at.row(n);
      else if constexpr (n < 2 * KS)
        f[n % A] = at.row(n - KS, C::BB);
      else if constexpr (n < 2 * KS + 2 * DB)
        f[n % A] = at.col((n - 2 * KS) / DB, (n - 2 * KS) % DB);
    };
    split_for<A>(fetch);
    floatx16 s = ZERO16, dp = ZERO16;
    DEERS_SPLIT_CHUNK_END();
    split_for<KS>([&](auto i) {
      constexpr int ks = decltype(i)::value;
      s = mfma_f16(f[ks % A], qf[ks], s);
      fetch(std::integral_constant<int, ks + A>());
      if constexpr (ks % 2 == 0) K.template request<ks>(next, ring + other);
      DEERS_SPLIT_CHUNK_END();
    });
    if (kb == qb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) > (lane & 31)) s[r] = -INFINITY;
    }
    DEERS_SPLIT_CHUNK_END();
    split_for<KS>([&](auto i) {
      constexpr int ks = decltype(i)::value, R = 16 / KS;
      dp = mfma_f16(f[(KS + ks) % A], dof[ks], dp);
      fetch(std::integral_constant<int, KS + ks + A>());
      if constexpr (ks % 2 == 0) V.template request<ks>(next, ring + other + C::BB);
#pragma unroll
      for (int r = R * ks; r < R * ks + R; ++r) s[r] = fast_exp2(fmaf(s[r], c, lse2));
      DEERS_SPLIT_CHUNK_END();
    });
    half8 ds[2];
#pragma unroll
    for (int r = 0; r < 8; ++r) s[r] *= dp[r] + nd;
    ds[0] = pack_regs(s, 0);
    DEERS_SPLIT_CHUNK_END();
    split_for<2 * DB>([&](auto i) {
      constexpr int n = decltype(i)::value, ms = n / DB, db = n % DB;
      dq[0][db] = mfma_f16(f[(2 * KS + n) % A], ds[ms], dq[0][db]);
      fetch(std::integral_constant<int, 2 * KS + n + A>());
      if constexpr (n < DB) {  // the other half of dS
        constexpr int R = 8 / DB;
#pragma unroll
        for (int r = 8 + R * n; r < 8 + R * n + R; ++r) s[r] *= dp[r] + nd;
        if constexpr (n == DB - 1) ds[1] = pack_regs(s, 1);
      }
      DEERS_SPLIT_CHUNK_END();
    });
    at.move(other - slot);
    slot = other;
  }
  half_t* const row = (half_t*)p.dq + b_ * p.sdq.b + h_ * p.sdq.h + (int64_t)qread * p.sdq.t;
  const float mul = p.scale;
  settle_loads();  // the zeros that the last stage asked for
  settle_lds_reads();
  SplitMerge<D, W>::leave(dq, ring, lane);
  SplitMerge<D, W>::template gather<1, false, 4 * C::BB>(dq, lds_address(smem), nullptr, &mul, &row, qrow < T, wave, lane);
}

template <int D, int W, bool SCALED_Q>
__device__ __forceinline__ void split_dkdv_body(const BwdParams& p, int bh, int kb, int n_blocks, char* smem, int wave,
                                                int lane) {
  using C = SplitCfg<D>;
  constexpr int KS = C::KS, DB = C::DB, A = kSplitAhead;
  const int g = lane >> 5, T = p.T;
  const int b_ = bh / p.H, h_ = bh % p.H;
  const int krow = 32 * kb + (lane & 31), kread = min(krow, T - 1);
  const uint32_t ring = lds_address(smem) + wave * 4 * C::BB;
  const uint32_t resident = lds_address(smem) + 2 * C::BB;  // wave 0's second slot: K, V
  float* stat = (float*)(smem + W * 4 * C::BB) + wave * kSplitStat<D>;

  half8 kf[KS], vf[KS];
  if constexpr (kSplitDirect<D>) {
    split_global_frags<D>(kf, p.k, p.sk, b_, h_, 32 * kb, T, lane);
    split_global_frags<D>(vf, p.v, p.sv, b_, h_, 32 * kb, T, lane);
  } else {
    split_load_resident<D, W>(p.k, p.sk, p.v, p.sv, b_, h_, 32 * kb, T, resident, wave, lane);
  }
  const SplitStream<D> Q(p.q, p.sq, b_, h_, T, lane), dO(p.d_o, p.sdo, b_, h_, T, lane);
  const SplitRowDots<D> dots(p.so, T, lane);
  const rsrc_t o_rsrc = dots.rsrc(p.o, p.so, b_, h_, T);
  half8 o[C::NI];
  const float* lse = p.lse + (int64_t)bh * T;
  float lse_row = 0.f;
  int qb = kb + wave;
  if (qb < n_blocks) {
    Q.request_all(qb, p.q, p.sq, b_, h_, T, ring, lane);
    dO.request_all(qb, p.d_o, p.sdo, b_, h_, T, ring + C::BB, lane);
#pragma unroll
    for (int i = 0; i < C::NI; ++i) o[i] = dots.load(o_rsrc, i, qb);
    lse_row = lse[min(32 * qb + (lane & 31), T - 1)];
  }
  const float c = SCALED_Q ? 1.f : p.scale_log2;
  floatx16 acc[2][DB];  // dK, dV
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = acc[1][db] = ZERO16;
  settle_loads();
  if constexpr (!kSplitDirect<D>) {
    __syncthreads();
    const SplitFrags<D> at(resident, lane);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = at.row(ks);
      vf[ks] = at.row(ks, C::BB);
    }
    settle_lds_reads();
    __syncthreads();  // the second slots are free
  }

  SplitFrags<D> at(ring, lane);
  uint32_t slot = 0;
  for (; qb < n_blocks; qb += W) {
    settle_loads();
    const uint32_t other = slot ^ (2 * C::BB);
    const int next = min(qb + W, n_blocks);
    // -LSE * log2(e), one row per lane, to the rows the accumulators hold; padded queries' probabilities are zero
    stat[lane & 31] = 32 * qb + (lane & 31) < T ? -lse_row * kLog2e : -INFINITY;
    // fragments in the order of their use: Q rows, dO rows, dO columns, Q columns
    half8 f[A], lin[2];
    const uint32_t lin_at = opaque(ring + slot + C::BB + lane * 16);
    auto fetch = [&](auto i) {
      constexpr int n = decltype(i)::value, m = n - 2 * KS;
      if constexpr (n < KS)
        f[n % A] = at.row(n);
      else if constexpr (n < 2 * KS)
        f[n % A] = at.row(n - KS, C::BB);
      else if constexpr (m < 4 * DB)
        f[n % A] = at.col(m % (2 * DB) / DB, m % DB, m < 2 * DB ? C::BB : 0);
    };
    split_for<A>(fetch);
    if constexpr (D != 32) {
#pragma unroll
      for (int i = 0; i < 2; ++i) lin[i] = lds_read_half8_at(lin_at + i * C::LB);
    }
    float bias[16];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 b = *(const floatx4*)(stat + 8 * r4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[4 * r4 + e] = b[e];
    }
    typename SplitRowDots<D>::Part parts[C::NI];
    floatx16 s = ZERO16, dp = ZERO16;
    DEERS_SPLIT_CHUNK_END();
    split_for<KS>([&](auto i) {
      constexpr int ks = decltype(i)::value;
      if (SCALED_Q) scale_frags<1>(&f[ks % A], p.scale_log2);
      s = mfma_f16(f[ks % A], kf[ks], s);
      if constexpr (D != 32) fetch(std::integral_constant<int, ks + A>());
      if constexpr (ks % 2 == 0) Q.template request<ks>(next, ring + other);
      parts[ks] = dots.multiply(o[ks], D == 32 ? f[(KS + ks) % A] : lin[ks & 1]);
      if constexpr (D == 32) fetch(std::integral_constant<int, ks + A>());
      if constexpr (D != 32 && ks + 2 < C::NI) lin[ks & 1] = lds_read_half8_at(lin_at + (ks + 2) * C::LB);
      if constexpr (ks == KS - 1) dots.leave(stat + 64, parts, lane);
      DEERS_SPLIT_CHUNK_END();
    });
    if (qb == kb) {  // queries of the diagonal block that come before the key
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) < (lane & 31)) s[r] = -INFINITY;
    }
    lse_row = lse[min(32 * next + (lane & 31), T - 1)];
    DEERS_SPLIT_CHUNK_END();
    split_for<KS>([&](auto i) {
      constexpr int ks = decltype(i)::value, R = 16 / KS;
      dp = mfma_f16(f[(KS + ks) % A], vf[ks], dp);
      fetch(std::integral_constant<int, KS + ks + A>());
      if constexpr (ks % 2 == 0) dO.template request<ks>(next, ring + other + C::BB);
#pragma unroll
      for (int r = R * ks; r < R * ks + R; ++r) s[r] = fast_exp2(fmaf(s[r], c, bias[r]));
      if constexpr (ks == (KS > 2 ? 1 : 0)) {
        stat[32 + (lane & 31)] = -dots.sum(stat + 64, parts, lane);
      }
      DEERS_SPLIT_CHUNK_END();
    });
    half8 pf[2];
    pf[0] = pack_regs(s, 0);
    float nd[16];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 b = *(const floatx4*)(stat + 32 + 8 * r4 + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) nd[4 * r4 + e] = b[e];
    }
    DEERS_SPLIT_CHUNK_END();
    // dV, then dK
    split_for<4 * DB>([&](auto i) {
      constexpr int m = decltype(i)::value, n = m % (2 * DB), ms = n / DB, db = n % DB;
      if constexpr (m < 2 * DB)
        acc[1][db] = mfma_f16(f[(2 * KS + m) % A], pf[ms], acc[1][db]);
      else
        acc[0][db] = mfma_f16(f[(2 * KS + m) % A], pf[ms], acc[0][db]);
      fetch(std::integral_constant<int, 2 * KS + m + A>());
      if constexpr (m < C::NI) o[m] = dots.load(o_rsrc, m, next);
      if constexpr (m == 0) pf[1] = pack_regs(s, 1);
      if constexpr (m >= DB && m < 2 * DB) {
        constexpr int R = 16 / DB;
#pragma unroll
        for (int r = R * (m - DB); r < R * (m - DB) + R; ++r) dp[r] = (dp[r] + nd[r]) * s[r];
        if constexpr (m == 2 * DB - 1) pf[0] = pack_regs(dp, 0);
      }
      if constexpr (m == 2 * DB) pf[1] = pack_regs(dp, 1);
      DEERS_SPLIT_CHUNK_END();
    });
    at.move(other - slot);
    slot = other;
  }
  half_t* const row[2] = {(half_t*)p.dk + b_ * p.sdk.b + h_ * p.sdk.h + (int64_t)kread * p.sdk.t,
                          (half_t*)p.dv + b_ * p.sdv.b + h_ * p.sdv.h + (int64_t)kread * p.sdv.t};
  const float mul[2] = {p.scale, 1.f};
  settle_loads();  // the zeros that the last stage asked for
  settle_lds_reads();
  SplitMerge<D, W>::leave(acc, ring, lane);
  SplitMerge<D, W>::template gather<2, false, 4 * C::BB>(acc, lds_address(smem), nullptr, mul, row, krow < T, wave, lane);
}
#undef DEERS_SPLIT_CHUNK_END

// Ranks alternate between the roles, longest first: rank 2 r is the dK/dV block of keys 32 r ..,
// rank 2 r + 1 the dQ block as many rows from the end.
template <int D, int W, bool SCALED_Q>
__global__ __launch_bounds__(64 * W, D == 128 ? 1 : 2) void attn_bwd_f16_split_kernel(BwdParams p, int BH, int n_blocks) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  fetch_arguments<decltype(attn_bwd_f16_split_kernel<D, W, SCALED_Q>)>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bh, rank;
  if (!map_block_even(blockIdx.x, 2 * n_blocks, BH, &bh, &rank)) return;
  if (rank & 1)
    split_dq_body<D, W, SCALED_Q>(first_argument<BwdParams>(), bh, n_blocks - 1 - (rank >> 1), n_blocks, smem, wave, lane);
  else
    split_dkdv_body<D, W, SCALED_Q>(first_argument<BwdParams>(), bh, rank >> 1, n_blocks, smem, wave, lane);
}

template <int D, int W, bool DOUBLE>
void launch_fwd_split(const FwdParams& p, int BH, bool scaled_q, hipStream_t stream) {
  const auto kernel = attn_fwd_f16_split_kernel<D, W, DOUBLE>;
  constexpr size_t lds = split_fwd_lds<D, W, DOUBLE>();
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  const int grid = map_even_blocks(n_blocks, BH);
  // even CU totals at D = 128 (15 x 777 10.6 -> 10.3 us, 9 x 1500 15.2 -> 14.6); below it the launch is the chain of its
  // longest wave, which should start first (9 x 1500 x 64 10.3 -> 11.0)
  static PairedState paired;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * W), lds, stream, p, BH, n_blocks,
                     D == 128 ? paired_cus(paired, kernel, 64 * W, lds, grid) : 0, (int)scaled_q);
}
template <int D, int W, bool SCALED_Q = false>
void launch_bwd_split(const BwdParams& p, int BH, hipStream_t stream) {
  const auto kernel = attn_bwd_f16_split_kernel<D, W, SCALED_Q>;
  constexpr size_t lds = split_bwd_lds<D, W>();
  static bool attr_set = false;
  if (!attr_set) allow_lds(kernel, lds);
  attr_set = true;
  const int n_blocks = (p.T + 31) / 32;
  hipLaunchKernelGGL(kernel, dim3(map_even_blocks(2 * n_blocks, BH)), dim3(64 * W), lds, stream, p, BH, n_blocks);
}

}  // namespace

// Which launches come here and in which form, fitted to times of both directions in every form and of the 128-row
// kernels at T = 32 .. 4096 and some 20 numbers of heads each, per head width (the waves: 1300 launches; the lines below:
// 2500).  nb = T / 32 is the length of a walk, n = heads * nb the number of workgroups, u = n * D / 64 their number
// weighted by what a block of the other operand weighs.
//
// Waves: four while the workgroups are few and for long walks, since a walk of nb blocks is nb / W stages long; fewer
// where the device is full anyway and every wave costs its start and the merge (us in 4 / 2 / 1 waves, forward D = 64:
// 12 x 512 5.8 / 7.7 / 11.1, 62 x 512 11.6 / 9.1 / 12.3, 200 x 256 11.5 / 11.0 / 8.8; backward D = 128: 6 x 768
// 14.2 / 20.3 / 31.6, 15 x 1024 40.4 / 32.0 / 46.2, 187 x 256 73.4 / 49.0 / 38.3).  Twice the blocks in LDS where a CU has
// one workgroup or two (forward D = 128, once / twice: 10 x 512 6.8 / 6.7, 6 x 128 4.7 / 4.5, 15 x 777 10.8 / 11.9; D = 32
// 8 x 2038 9.4 / 8.6, 12 x 1500 7.9 / 7.4, 5 x 4096 16.7 / 15.8, 12 x 2048 10.4 / 10.7).  The
// forward at D = 32: four up to some 90 heads, walks of three blocks included, and two up to 250, of two blocks up to
// 120 (us in 4 / 2 / 1: 50 x 86 3.0 / 3.4 / 3.5, 120 x 54 3.0 / 3.0 / 3.2, 130 x 54 3.4 / 3.4 / 3.2, 240 x 86 4.2 / 3.6 /
// 3.8, 90 x 246 4.4 / 4.8 / 5.9, 250 x 150 5.6 / 4.6 / 4.9, 300 x 150 6.1 / 5.3 / 5.1).
//
// Takes, us in the 128-row kernels / these: walks of up to 15 blocks nearly always (those form 128 rows where 64 to 384
// are, and every stage has a barrier: forward 419 x 96 x 64 8.3 / 5.5, 286 x 300 x 128 28.4 / 22.1, 327 x 400 x 64 24.9 / 19.2;
// backward 403 x 160 x 128 73.9 / 48.3, 179 x 320 x 64 26.5 / 21.7, 107 x 416 x 64 25.0 / 21.8) until the operands no longer
// stay in the L2 beside each other (forward 1043 x 256 x 64 34.1 / 41.2, backward 723 x 256 x 64 69.4 / 91.4); longer ones
// while the 128-row kernels leave CUs idle, since each of the waves reading all of the other operand for 32 rows costs
// more than it saves elsewhere (forward 24 x 2048 x 32 21.0 / 17.2, 13 x 3000 x 64 34.6 / 31.1, 10 x 4096 x 128 64.3 / 69.8,
// 20 x 3000 x 64 37.2 / 41.4; backward 9 x 2048 x 64 44.9 / 31.9, 9 x 4096 x 64 105.7 / 100.6, 12 x 3000 x 128 144.7 / 157.6,
// 20 x 2048 x 64 56.4 / 62.3).  Seven or eight heads give each XCD one, which is what those kernels like best (backward 8 x
// 3000 x 64 51.2 / 56.5, 9 x 3000 x 64 63.8 / 62.9).  At nb = 12 to 16 they are as fast or faster while all their
// workgroups are resident two to a CU (forward 168 x 512 x 64 14.8 / 15.8, 80 x 512 x 128 15.5 /
// 17.5, 124 x 372 x 64 10.6 / 11.8, but 108 x 372 x 64 10.3 / 9.7, 148 x 372 x 64 12.3 / 11.3).
// The forward takes what the backward takes: then both form their scores from Q itself.
// At D = 32 from 16 blocks on the forward's line lies where its error does, not its time: the 128-row kernel's reference moves
// late and P is rounded against it (O from 64 bits, 128 rows / here: 31 x 2425 3.24e-4 / 3.12e-4, 75 x 1024 3.27e-4 / 3.11e-4; us
// 23.6 / 26.2, 12.8 / 14.4).  At 16 blocks the backward comes along: 120 x 512 8.5 / 9.5, with it 26.8 / 24.3.
extern bool attn_128_rows;  // runtime.hip
struct SplitSize {
  int64_t nb, u;
  SplitSize(int64_t BH, int64_t T, int64_t D) : nb((T + 31) / 32), u(BH * nb * D / 64) {}
};
// By head width: 32, 64, 128.
static int64_t of_width(int64_t D, int64_t w32, int64_t w64, int64_t w128) { return D == 32 ? w32 : D == 64 ? w64 : w128; }
// Up to `low`, and again from `again` up to `most`.
static bool outside(int64_t u, int64_t low, int64_t again, int64_t most) { return u <= low || (u > again && u <= most); }
bool attn_fwd_f16_split_takes(int64_t BH, int64_t T, int64_t D) {
  if (attn_128_rows) return false;
  const SplitSize z(BH, T, D);
  const int64_t nb = z.nb, u = z.u;
  if (nb <= 2) return u <= of_width(D, 5000, 5000, 9000);
  if (nb <= 4) return u <= of_width(D, 4500, 5200, 6400);
  if (nb <= 8) return u <= of_width(D, 5000, 5800, 8400);
  if (nb <= 11) return u <= of_width(D, 4500, 6000, 8000);
  if (nb <= 12) return outside(u, of_width(D, 4500, 1350, 2048), of_width(D, 4500, 1660, 3300), of_width(D, 4500, 5800, 7000));
  if (nb <= 15) return outside(u, of_width(D, 4000, 6800, 2048), 3300, of_width(D, 4000, 6800, 7500));
  if (nb <= 16) return outside(u, of_width(D, 1200, 1300, 2048), of_width(D, 1540, 3000, 8192), of_width(D, 4200, 5800, 8192));
  return u <= of_width(D, 1200, 1200, 2048);
}
bool attn_bwd_f16_split_takes(int64_t BH, int64_t T, int64_t D) {
  if (!attn_fwd_f16_split_takes(BH, T, D)) return false;
  const SplitSize z(BH, T, D);
  const int64_t nb = z.nb, u = z.u;
  if (nb <= 2) return u <= of_width(D, 4000, 4000, 8600);
  if (nb <= 3) return u <= of_width(D, 3600, 4300, 8600);
  if (nb <= 4) return u <= of_width(D, 3600, 3500, 6400);
  if (nb <= 6) return u <= of_width(D, 4000, 3800, 6200);
  if (nb <= 8) return u <= of_width(D, 3600, 3000, 4700);
  if (nb <= 11) return u <= of_width(D, 2600, 3600, 5000);
  if (nb <= 12) return u <= of_width(D, 2600, 2900, 4400);
  if (nb <= 15) return u <= of_width(D, 3200, 3400, 4700);
  if (nb <= 16) return u <= of_width(D, 3200, 1300, 2048);
  if (nb <= 20) return u <= of_width(D, 700, 1000, 1200);
  if (nb <= 23) return u <= of_width(D, 760, 1000, 1200);
  if (nb < 72) return u <= of_width(D, 720, 960, 1200);
  if (BH > 6 && BH <= 8) return u <= of_width(D, 700, 640, 1110);
  return u <= of_width(D, 700, 1100, 1700);
}
static int waves(const SplitSize& z, int64_t four, int64_t two, int64_t shortest = 4) {
  return z.u <= four && z.nb >= shortest ? 4 : z.u <= std::max(four, two) && z.nb >= 2 ? 2 : 1;
}
static int fwd_waves(const SplitSize& z, int64_t D) {
  const int64_t nb = z.nb, sq = nb * nb;
  const int64_t four = of_width(D, (nb < 5 ? 45 : 50) * nb, std::min(90 * nb, 700 + 25 * nb), std::min(160 * nb, 780 + 27 * nb));
  const int64_t two = of_width(D, nb < 3 ? 120 : std::min<int64_t>(125 * nb, 900), std::min<int64_t>(64 * sq, 1700),
                               std::min(120 * sq, 1300 + 60 * nb));
  return waves(z, four, nb > 16 ? z.u : two, D == 32 ? 3 : 4);
}
static bool fwd_twice(const SplitSize& z, int64_t D) { return z.u <= of_width(D, 340, 256, 448); }
static int bwd_waves(const SplitSize& z, int64_t D) {
  const int64_t nb = z.nb;
  const int64_t four = of_width(D, std::min(24 * nb, 120 + 9 * nb), std::min(32 * nb, 160 + 12 * nb), std::max<int64_t>(256, 72 + 20 * nb));
  return waves(z, std::min<int64_t>(four, 768), of_width(D, 40 * nb, 80 * nb, 400 + 60 * nb));
}

template <int D, int W>
static void launch_fwd(const FwdParams& p, int BH, bool twice, bool scaled_q, hipStream_t stream) {
  if constexpr (W == 4) {
    if (twice) return launch_fwd_split<D, W, true>(p, BH, scaled_q, stream);
  }
  launch_fwd_split<D, W, false>(p, BH, scaled_q, stream);
}
template <int D>
static void launch_fwd(const FwdParams& p, int BH, bool scaled_q, hipStream_t stream) {
  const SplitSize z(BH, p.T, D);
  const int w = fwd_waves(z, D);
  const bool twice = w >= 4 && fwd_twice(z, D);
  if (w >= 4)
    launch_fwd<D, 4>(p, BH, twice, scaled_q, stream);
  else if (w >= 2)
    launch_fwd<D, 2>(p, BH, twice, scaled_q, stream);
  else
    launch_fwd<D, 1>(p, BH, twice, scaled_q, stream);
}
// Scaled queries: captured launches that the 128-row kernel would have, larger than what comes here in four waves (in
// four 300 x 256 x 128 119.7 us, in one 67.3; 30 x 1300 x 128 in four 109.6, in two 88.0).
template <int D>
static void launch_bwd(const BwdParams& p, int BH, bool from_q, hipStream_t stream) {
  const int w = bwd_waves(SplitSize(BH, p.T, D), D);
  if (!from_q && w >= 2)
    launch_bwd_split<D, 2, true>(p, BH, stream);
  else if (!from_q)
    launch_bwd_split<D, 1, true>(p, BH, stream);
  else if (w >= 4)
    launch_bwd_split<D, 4>(p, BH, stream);
  else if (w >= 2)
    launch_bwd_split<D, 2>(p, BH, stream);
  else
    launch_bwd_split<D, 1>(p, BH, stream);
}

void launch_attn_fwd_f16_split(const FwdParams& p, int B, int D, bool from_q, hipStream_t stream) {
  LaunchScope scope("attn_fwd_f16", stream);
  switch (D) {
    case 32: launch_fwd<32>(p, B * p.H, !from_q, stream); break;
    case 64: launch_fwd<64>(p, B * p.H, !from_q, stream); break;
    case 128: launch_fwd<128>(p, B * p.H, !from_q, stream); break;
  }
}
void launch_attn_bwd_f16_split(const BwdParams& p, int B, int D, bool from_q, hipStream_t stream) {
  LaunchScope scope("attn_bwd_f16", stream);
  switch (D) {
    case 32: launch_bwd<32>(p, B * p.H, from_q, stream); break;
    case 64: launch_bwd<64>(p, B * p.H, from_q, stream); break;
    case 128: launch_bwd<128>(p, B * p.H, from_q, stream); break;
  }
}

}  // namespace deers
