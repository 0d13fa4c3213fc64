// Decode attention: one query row per (b,h) against a KV cache of L rows, f16.
//
// Same math as the forward with tgt_len = 1 and seqlen_offset = L-1, where the
// causal mask row is all zero (src/nn/functional.rs:26,42).  1 FLOP per byte:
// the kernel is an HBM stream, so the design is about bytes in flight, not
// matrix cores.
//
//   A workgroup streams `chunk` cache rows of one head.
//   A row of D halfs is covered by LPR = D/8 lanes with one 16-byte load each,
//   so a wave reads 1 KiB of K and 1 KiB of V per load instruction, fully
//   coalesced.  A tile is kDecRowsPerIt rows per lane group, K and V loads
//   issued together (V does not wait for the scores), the first ones before the query is
//   worked on.  A workgroup that has a CU to itself requests the next tile before it works
//   on the one at hand (PIPELINED); where a CU holds several workgroups, each one's
//   computation already overlaps the others' loads and the second tile only adds
//   requests that compete (32 x 12 heads x 4096 x 64: 60.9 us without, 63.9 with;
//   16 x 12 x 700: 10.2 without, 9.5 with).
//   Each lane group keeps a private online softmax (m, l, o[8] per lane) over
//   the rows it visits; the groups of a wave are merged by lane exchanges that
//   leave every lane its own columns, the waves through LDS, all in a fixed order.
//   With one split per head the workgroup writes the f16 output itself.  Otherwise
//   the split's partial (m, l, o[D]) goes to the workspace and the last split of the head
//   to arrive merges them in split order; the splits of a head are given to one XCD, whose
//   L2 is where they meet.  (A merge across XCDs was tried: the device-scope fences it
//   needs cost several times the whole stream.)  Where the splits may not share an
//   XCD a second tiny kernel merges: same order, same bits.
//   us per call, against a split into 256 / heads rounded up to a power of two, no early
//   loads and the merge always a launch of its own: 12 heads x 1500 x 64
//   8.95 -> 6.1, 12 x 6000 x 64 13.9 -> 9.6, 48 x 1000 x 64 9.9 -> 7.1, 24 x 900 x 128 13.9 -> 7.3,
//   4 x 16000 x 64 19.8 -> 9.9 (3.3 TB/s).
//
//   Append form (a generation step): instead of a ready query the kernel takes the new
//   token's q, k, v projections, rotates q and k at the token's position (the
//   arithmetic of decode_qkv_kernel: f32, one rounding to f16), writes k and v to cache
//   row L and attends over rows [0, L] -- rows [0, L) streamed from the cache, row L from
//   the registers that hold it, so nothing written by this launch is read back from
//   memory.  One launch per block and step instead of two.
#include <algorithm>

#include "common.h"

namespace deers {

constexpr int kDecRowsPerIt = 4;  // cache rows of a lane group's tile
constexpr int kDecSplitRows = 128;  // a split's smallest share of the cache

// Number of splits per head: as many as the head's XCD has CUs for its heads (32 CUs, heads dealt
// to 8 XCDs), each with about kDecSplitRows rows or more.  Beyond one workgroup per CU a split is only
// another start-up and another partial to merge (12 heads x 6000 x 64: 9.6 us in 16 splits, 10.5
// in 21, 13.9 in 47); below kDecSplitRows rows the merge costs what the shorter stream saves
// (12 x 1500 x 64: 6.1 us in 12 splits, 9.1 in 24).
// Where that leaves three CUs of ten without a workgroup (11 heads of an XCD in two splits, 17 to 21 in
// one) a CU gets two, if the caches are long enough for the stream to be what counts (us in one per CU /
// two per CU: 132 x 1024 x 64 10.1 / 9.8, 132 x 8192 x 64 54.6 / 44.6, 160 x 8192 x 64 56.3 / 50.3, 88 x 8192 x 128 60.1 /
// 54.8; but 160 x 768 x 64 8.7 / 9.0).  With fewer idle ones it gains nothing (12 heads, three of four CUs:
// 96 x 16384 x 64 60.9 / 59.9).
// Spreading fewer than eight heads over all XCDs, to be merged by a second launch, gains only beyond any
// cache of interest (2 x 65536 x 64: 19.5 us on two XCDs, 17.4 on eight; 2 x 16384: 9.0 / 13.6).
int decode_pick_splits(int64_t BH, int64_t L, int64_t D, int* chunk) {
  const int64_t heads = (BH + 7) / 8, by_rows = (L + kDecSplitRows - 1) / kDecSplitRows;
  int64_t by_cus = 32 / heads;
  if (L * D >= 65536 && 10 * heads * by_cus < 7 * 32 && 64 / heads > 2 * by_cus) by_cus = 64 / heads;
  const int64_t want = std::max<int64_t>(1, std::min(by_cus, by_rows));
  const int64_t c = std::max<int64_t>(16, ((L + want - 1) / want + 15) / 16 * 16);
  *chunk = (int)c;
  return (int)std::max<int64_t>(1, (L + c - 1) / c);  // no split without rows
}

// The thread's 8 columns (8*part ..) of rotate_half RoPE applied to one [D] row: columns
// below D/2 are x1*cos + x2*sin, the others x2*cos - x1*sin, with x1 / x2 the lower /
// upper half's elements of the same index (src/models/gpt.rs:49-73).
struct RotateIn { half8 lower, upper; };  // the two halves' elements of the thread's columns
template <int D>
__device__ __forceinline__ RotateIn rotate_load(const half_t* row, int part) {
  const int c = 8 * part % (D / 2);
  return {*(const half8*)(row + c), *(const half8*)(row + c + D / 2)};
}
template <int D>
__device__ __forceinline__ half8 rotate_row(const RotateIn& x, half8 cs, half8 sn, int part) {
  const bool upper = 8 * part >= D / 2;
  half8 out;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x1 = (float)x.lower[e], x2 = (float)x.upper[e], co = (float)cs[e], si = (float)sn[e];
    out[e] = upper ? (half_t)(x2 * co - x1 * si) : (half_t)(x1 * co + x2 * si);
  }
  return out;
}

// One step of the sum over a wave's row groups: the lane and its partner `off` away add up their
// column sums, each for one half of the 2 * KEEP columns they share; `col` is the first it keeps.
template <int KEEP>
__device__ __forceinline__ void halve_columns(float (&o)[8], int off, int lane, int& col) {
  const bool hi = lane & off;
  col += hi ? KEEP : 0;
#pragma unroll
  for (int e = 0; e < KEEP; ++e) {
    const float mine = hi ? o[e + KEEP] : o[e], theirs = hi ? o[e] : o[e + KEEP];
    o[e] = mine + __shfl_xor(theirs, off, 64);
  }
}

// Sum over the splits of a head in split order, for column d.  The partials were written by other
// workgroups of the same XCD or by an earlier launch, so they are read past the CU's own cache;
// kMergeBatch splits' loads are in flight at once.
constexpr int kMergeBatch = 8;
template <int D>
__device__ __forceinline__ half_t merge_splits(const DecodeParams& p, int bh, int d) {
  const float* ml = p.part_ml + (int64_t)bh * p.splits * 2;
  const float* po = p.part_o + (int64_t)bh * p.splits * D + d;
  float M = -INFINITY, lsum = 0.f, osum = 0.f;
  for (int s0 = 0; s0 < p.splits; s0 += kMergeBatch) {
    float ms[kMergeBatch], ls[kMergeBatch], os[kMergeBatch];
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const int s = min(s0 + u, p.splits - 1);
      ms[u] = __hip_atomic_load(ml + 2 * s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ls[u] = __hip_atomic_load(ml + 2 * s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      os[u] = __hip_atomic_load(po + (int64_t)s * D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float m_new = M;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) m_new = fmaxf(m_new, ms[u]);  // repeats of the last split change no maximum
    const float alpha = fast_exp2(M - m_new);  // every split saw a row: m_new is finite
    lsum *= alpha;
    osum *= alpha;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float w = s0 + u < p.splits ? fast_exp2(ms[u] - m_new) : 0.f;
      lsum += w * ls[u];
      osum += w * os[u];
    }
    M = m_new;
  }
  return (half_t)(osum / lsum);
}

template <int D, bool APPEND, bool PIPELINED>
__global__ __launch_bounds__(256) void attn_decode_f16_kernel(DecodeParams p) {
  constexpr int LPR = D / 8;            // lanes per cache row
  constexpr int GROUPS = 256 / LPR;     // row groups per workgroup
  constexpr int TILE = GROUPS * kDecRowsPerIt;
  constexpr int WAVES = 4;
  __shared__ float red_m[WAVES];
  __shared__ float red_l[WAVES];
  __shared__ float red_o[WAVES * D];
  __shared__ int last_flag;

  const int tid = threadIdx.x, lane = tid & 63;
  const int part = tid % LPR;
  const int grp = tid / LPR;
  // the splits of a head share block id % 8, that is, an XCD
  const int bh = (int)(blockIdx.x >> 3) / p.splits * 8 + (int)(blockIdx.x & 7);
  const int split = (int)(blockIdx.x >> 3) % p.splits;
  if (bh >= p.BH) return;
  const int b = bh / p.H, h = bh % p.H;

  const half_t* K = (const half_t*)p.k + b * p.skb + h * p.skh + 8 * part;
  const half_t* V = (const half_t*)p.v + b * p.skb + h * p.skh + 8 * part;
  const int row_begin = split * p.chunk;
  const int row_end = min(row_begin + p.chunk, p.L);

  // One tile: kDecRowsPerIt rows of K and of V per lane group.  Rows past the end repeat the last
  // one (their scores are masked).  Every cache byte is used once: non-temporal loads keep the
  // stream from displacing itself in the caches and measurably raise the achieved HBM rate.
  struct Tile { half8 k[kDecRowsPerIt], v[kDecRowsPerIt]; };
  auto load = [&](Tile& t, int r0) {
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) {
      const int64_t off = (int64_t)min(r0 + grp + u * GROUPS, row_end - 1) * p.skl;
      t.k[u] = __builtin_nontemporal_load((const half8*)(K + off));
      t.v[u] = __builtin_nontemporal_load((const half8*)(V + off));
    }
  };
  // What the query needs is requested before the first tile, which is on its way while the query is
  // worked on (the other order makes the rotation wait for the tile: 32 x 12 x 600 x 64, appending,
  // 14.5 us against 13.7).  The new row is handled by one lane group of the last split.
  half8 qh = {0, 0, 0, 0, 0, 0, 0, 0}, k_new = qh, v_new = qh, cs = qh, sn = qh;
  const bool owns_new_row = APPEND && grp == 0 && split == p.splits - 1;
  const int64_t in_off = b * p.in_b + h * p.in_h;
  RotateIn q_raw{qh, qh}, k_raw{qh, qh};
  if constexpr (APPEND) {
    const int c = 8 * part % (D / 2);
    q_raw = rotate_load<D>((const half_t*)p.q_in + in_off, part);
    cs = *(const half8*)((const half_t*)p.cos_row + c);
    sn = *(const half8*)((const half_t*)p.sin_row + c);
    if (owns_new_row) {
      k_raw = rotate_load<D>((const half_t*)p.k_in + in_off, part);
      v_new = *(const half8*)((const half_t*)p.v_in + in_off + 8 * part);
    }
  } else {
    qh = *(const half8*)((const half_t*)p.q + (int64_t)bh * D + 8 * part);
  }
  Tile cur, nxt;
  if (row_begin < row_end) load(cur, row_begin);
  if constexpr (APPEND) {
    qh = rotate_row<D>(q_raw, cs, sn, part);
    if (owns_new_row) {
      k_new = rotate_row<D>(k_raw, cs, sn, part);
      *(half8*)(const_cast<half_t*>(K) + (int64_t)p.L * p.skl) = k_new;
      *(half8*)(const_cast<half_t*>(V) + (int64_t)p.L * p.skl) = v_new;
    }
  }
  float qf[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) qf[e] = (float)qh[e] * p.scale_log2;

  float m = -INFINITY, l = 0.f;
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  if (owns_new_row) {  // row L from registers, as the first row its lane group sees
    m = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) m += qf[e] * (float)k_new[e];
#pragma unroll
    for (int off = LPR / 2; off >= 1; off >>= 1) m += __shfl_xor(m, off, 64);
    l = 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (float)v_new[e];
  }

  auto attend = [&](const Tile& t, int r0) {
    float s[kDecRowsPerIt];
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) {
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc += qf[e] * (float)t.k[u][e];
#pragma unroll
      for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
      s[u] = (r0 + grp + u * GROUPS < row_end) ? acc : -INFINITY;
    }
    float m_new = m;
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) m_new = fmaxf(m_new, s[u]);
    // a lane group whose rows all lie past the end has seen nothing: keep its sums at zero
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = fast_exp2(m - m_ref);
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= alpha;
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) {
      const float pu = fast_exp2(s[u] - m_ref);
      l += pu;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += pu * (float)t.v[u][e];
    }
    m = m_new;
  };
  if constexpr (PIPELINED) {
    for (int r0 = row_begin; r0 < row_end; r0 += 2 * TILE) {
      if (r0 + TILE < row_end) load(nxt, r0 + TILE);
      attend(cur, r0);
      if (r0 + TILE < row_end) {
        if (r0 + 2 * TILE < row_end) load(cur, r0 + 2 * TILE);
        attend(nxt, r0 + TILE);
      }
    }
  } else {
    for (int r0 = row_begin; r0 < row_end; r0 += TILE) {
      attend(cur, r0);
      if (r0 + TILE < row_end) load(cur, r0 + TILE);
    }
  }

  // ---- merge the row groups (fixed order): within the wave by an exchange that halves the
  // columns a lane keeps at every step, so that in the end each lane holds the columns it will
  // write; then the four waves through LDS ----
  float wave_m = m;
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1) wave_m = fmaxf(wave_m, __shfl_xor(wave_m, off, 64));
  const float w = m == -INFINITY ? 0.f : fast_exp2(m - wave_m);
  l *= w;
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1) l += __shfl_xor(l, off, 64);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= w;
  int col = 8 * part;
  halve_columns<4>(o, 32, lane, col);
  halve_columns<2>(o, 16, lane, col);
  if constexpr (LPR <= 8) halve_columns<1>(o, 8, lane, col);
  if constexpr (LPR <= 4) o[0] += __shfl_xor(o[0], 4, 64);
  constexpr int COLS = D == 128 ? 2 : 1;  // columns per lane by now
  const int wave = tid >> 6;
#pragma unroll
  for (int e = 0; e < COLS; ++e) red_o[wave * D + col + e] = o[e];
  if (lane == 0) {
    red_m[wave] = wave_m;
    red_l[wave] = l;
  }
  __syncthreads();
  if (tid < D) {
    float M = red_m[0], lsum = 0.f, osum = 0.f;
#pragma unroll
    for (int wi = 1; wi < WAVES; ++wi) M = fmaxf(M, red_m[wi]);
#pragma unroll
    for (int wi = 0; wi < WAVES; ++wi) {
      const float ww = red_m[wi] == -INFINITY ? 0.f : fast_exp2(red_m[wi] - M);
      lsum += ww * red_l[wi];
      osum += ww * red_o[wi * D + tid];
    }
    if (p.splits == 1) {  // nothing to merge
      ((half_t*)p.o)[(int64_t)bh * D + tid] = (half_t)(osum / lsum);
      return;
    }
    const int64_t slot = (int64_t)bh * p.splits + split;
    p.part_o[slot * D + tid] = osum;
    if (tid == 0) {
      p.part_ml[slot * 2 + 0] = M;
      p.part_ml[slot * 2 + 1] = lsum;
    }
  }
  if (p.splits == 1 || !p.arrived) return;
  // The splits of a head share one XCD and so one L2: a completed store (vmcnt 0) is in that L2,
  // and relaxed device-scope atomics, which bypass the CU's own cache, are all the ordering
  // needed; no cache write-back or invalidation.
  wait_all_vmem();
  __syncthreads();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(p.arrived + bh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = before == p.splits - 1;
    if (last_flag)  // ready for the next launch
      __hip_atomic_store(p.arrived + bh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (last_flag && tid < D) ((half_t*)p.o)[(int64_t)bh * D + tid] = merge_splits<D>(p, bh, tid);
}

// The merge as a launch of its own, where the splits of a head may not meet in one L2.
template <int D>
__global__ __launch_bounds__(D) void attn_decode_merge_kernel(DecodeParams p) {
  const int bh = blockIdx.x, d = threadIdx.x;
  ((half_t*)p.o)[(int64_t)bh * D + d] = merge_splits<D>(p, bh, d);
}

void launch_attn_decode_f16(const DecodeParams& p, int B, int D, bool append, hipStream_t stream) {
  const dim3 grid(8 * p.splits * ((B * p.H + 7) / 8));  // a head's splits on one XCD: see the kernel
  {
    LaunchScope scope(append ? "attn_decode_append_f16" : "attn_decode_f16", stream);
    const bool alone = p.splits * p.BH <= 256;  // at most one workgroup per CU
#define DEERS_DECODE_CASE(DD, APP, PIPE)        \
  if (D == DD && append == APP && alone == PIPE) \
    hipLaunchKernelGGL((attn_decode_f16_kernel<DD, APP, PIPE>), grid, dim3(256), 0, stream, p);
    DEERS_DECODE_CASE(32, false, false)
    DEERS_DECODE_CASE(32, false, true)
    DEERS_DECODE_CASE(32, true, false)
    DEERS_DECODE_CASE(32, true, true)
    DEERS_DECODE_CASE(64, false, false)
    DEERS_DECODE_CASE(64, false, true)
    DEERS_DECODE_CASE(64, true, false)
    DEERS_DECODE_CASE(64, true, true)
    DEERS_DECODE_CASE(128, false, false)
    DEERS_DECODE_CASE(128, false, true)
    DEERS_DECODE_CASE(128, true, false)
    DEERS_DECODE_CASE(128, true, true)
#undef DEERS_DECODE_CASE
  }
  if (p.splits > 1 && !p.arrived) {
    LaunchScope scope("attn_decode_merge", stream);
    if (D == 32)
      hipLaunchKernelGGL(attn_decode_merge_kernel<32>, dim3(B * p.H), dim3(32), 0, stream, p);
    else if (D == 64)
      hipLaunchKernelGGL(attn_decode_merge_kernel<64>, dim3(B * p.H), dim3(64), 0, stream, p);
    else
      hipLaunchKernelGGL(attn_decode_merge_kernel<128>, dim3(B * p.H), dim3(128), 0, stream, p);
  }
}

}  // namespace deers
