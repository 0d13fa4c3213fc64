// Decode attention: one query row per (b,h) against a KV cache of L rows, f16.
//
// Same math as the forward with tgt_len = 1 and seqlen_offset = L-1, where the
// causal mask row is all zero (src/nn/functional.rs:26,42).  1 FLOP per byte:
// the kernel is an HBM stream, so the design is about bytes in flight, not
// matrix cores.
//
//   A workgroup streams a head's cache, or `chunk` rows of it.
//   A row of D halfs is covered by LPR = D/8 lanes with one 16-byte load each,
//   so a wave reads 1 KiB of K and 1 KiB of V per load instruction, fully
//   coalesced.  A tile is kDecRowsPerIt rows per lane group, the first one requested before
//   the query is worked on; the next tile's K is requested as soon as the scores are there, its V as
//   soon as the sums are.  A second tile's registers bring nothing (8 waves or 16 to a workgroup neither:
//   64 x 12 heads x 2000 x 64 57.9 us with 4, 57.9 with 8, 63.1 with 16), since by then the memory is what
//   bounds it: 6.4 to 6.8 TB/s from 60 MB on.
//   Each lane group keeps a private online softmax (m, l, o[8] per lane) over
//   the rows it visits; the groups of a wave are merged by lane exchanges that
//   leave every lane its own columns, the waves through LDS, all in a fixed order.
//   With one split per head the workgroup writes the f16 output itself.  Otherwise
//   the split's partial (m, l, o[D]) goes to the workspace and the last split of the head
//   to arrive merges them in split order; the splits of a head are given to one XCD, whose
//   L2 is where they meet.  (A merge across XCDs was tried: the device-scope fences it
//   needs cost several times the whole stream.)  Where the splits may not share an
//   XCD a second tiny kernel merges: same order, same bits.  It costs two microseconds more (12 heads
//   x 700 x 64 7.4 us, 4.8 in the launch; 12 x 6000 x 64 8.5 / 7.9).
//   A short call is a chain of latencies: the launch, its arguments, the query, the tile, the reductions, the meeting.  us per
//   call with lane exchanges through LDS, a wait for all of a tile before the next was requested, row addresses by 64-bit
//   products, arguments fetched where they are used and the partials read in batches of eight, and as it is: 12 heads x
//   200 x 64 4.4 -> 3.2, 12 x 1500 x 64 6.7 -> 5.8, 12 x 6000 x 64 9.0 -> 8.0, 112 x 2000 x 64 13.1 -> 12.1, 192 x 2000 x 64 18.6 ->
//   16.7; appending: 12 x 600 x 64 5.7 -> 4.7, 32 x 400 x 32 5.8 -> 4.2, 384 x 600 x 64 12.7 -> 11.7.
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
constexpr int kDecTile = 256 * 8 * kDecRowsPerIt;  // elements of K in a workgroup's tile
constexpr int kDecSplitRows = 128;  // a split's smallest share of the cache

// Number of splits per head: as many as the head's XCD has CUs for its heads (32 CUs, heads dealt
// to 8 XCDs), each with a tile or kDecSplitRows rows, whichever is more.  Beyond one workgroup per CU a split is only
// another start-up and another partial to merge (12 heads x 6000 x 64: 8.2 us in 16 splits, 8.6 in 8 and in 20;
// 24 x 1000 x 64: 6.2 us in 6, 6.6 in 8, 7.3 in 12); shorter than a tile it reads masked rows (8 heads x 4000 x 32: 5.3 us in
// 16 splits of a tile, 7.1 in 31).
// A cache of a few tiles stays whole, since the meeting of the splits takes as long as two tiles, and longer the
// more splits meet on an XCD (us whole / split: 12 x 200 x 64 3.8 / 4.3, 12 x 300 x 64 4.5 / 4.4; 56 x 500 x 64 5.3 / 5.5, 56 x
// 300 x 128 6.1 / 5.8; 88 x 500 x 64 5.5 / 5.9, 88 x 1000 x 64 8.4 / 7.5).
// Where that leaves three CUs of ten without a workgroup (11 heads of an XCD in two splits, 17 to 21 in
// one) a CU gets two, if the caches are long enough for the stream to be what counts (us in one per CU /
// two per CU: 136 x 2000 x 64 15.1 / 14.6, 136 x 4000 x 64 27.5 / 24.4, 160 x 4000 x 64 28.7 / 27.1; but 136 x 1000 x 64 8.9 / 9.4).
// With fewer idle ones it gains nothing (12 heads, three of four CUs).
// Spreading fewer than eight heads over all XCDs, to be merged by a second launch, gains only beyond any
// cache of interest (2 x 65536 x 64: 19.5 us on two XCDs, 17.4 on eight; 2 x 16384: 9.0 / 13.6).
int decode_pick_splits(int64_t BH, int64_t L, int64_t D, int* chunk) {
  const int64_t heads = (BH + 7) / 8, size = L * D, rows = std::max<int64_t>(kDecSplitRows, kDecTile / D);
  int64_t by_cus = 32 / heads;
  if (size >= 65536 && 10 * heads * by_cus < 7 * 32 && 64 / heads > 2 * by_cus) by_cus = 64 / heads;
  const int64_t whole = by_cus > 4 ? 2 : by_cus > 2 ? 4 : 5;
  const int64_t by_rows = size <= whole * kDecTile ? 1 : (L + rows - 1) / rows;
  const int64_t want = std::max<int64_t>(1, std::min(by_cus, by_rows));
  const int64_t c = std::max<int64_t>(16, ((L + want - 1) / want + 15) / 16 * 16);
  *chunk = (int)c;
  return (int)std::max<int64_t>(1, (L + c - 1) / c);  // no split without rows
}

// Heads of an XCD that one workgroup each attends over; the splits and the chunk of the others.  Where the heads fill
// the CUs once or more and up to half of them once again, the last ones are split as if they were alone, so that
// every CU gets a whole head and the same part of another one (us all whole / so: 264 x 400 x 64 8.5 / 7.4, 264 x 4000 x 64 54.9 / 42.1,
// 320 x 2000 x 64 30.4 / 27.5, 384 x 1000 x 64 17.4 / 16.8, 384 x 4096 x 64 63.6 / 62.4, 576 x 4000 x 64 96.7 / 86.6).  With more
// than half of them it loses (392 x 4000 x 64 62.7 / 64.6, 416 x 4000 x 64 64.5 / 68.1).
int decode_pick_whole(int64_t BH, int64_t L, int64_t D, int* splits, int* chunk) {
  const int64_t heads = (BH + 7) / 8, rest = heads % 32;
  const bool mixed = heads > 32 && rest > 0 && rest <= 16;
  *splits = decode_pick_splits(mixed ? 8 * rest : BH, L, D, chunk);
  return mixed && *splits > 1 ? (int)(heads - rest) : 0;
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

// Exchanges inside a wave on the vector unit (a shuffle through LDS takes some 120 clocks, and the ones of a tile follow
// each other: three for a row's score, six for the merge).
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), CTRL, 0xf, 0xf, true));
}
// The value of lane ^ OFF, OFF a multiple of 4.
template <int OFF>
__device__ __forceinline__ float from_lane_xor(float x) {
  if constexpr (OFF == 4) return __shfl_xor(x, 4, 64);
  if constexpr (OFF == 8) return dpp<0x128>(x);  // a row of 16 turned by 8
  const unsigned u = __float_as_uint(x);
  unsigned lo, hi;
  if constexpr (OFF == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    lo = r[0], hi = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    lo = r[0], hi = r[1];
  }
  // lo: the lower halves' values in both halves, hi: the upper halves'
  return __uint_as_float((threadIdx.x & OFF) ? lo : hi);
}
// Sum / maximum over the LANES lanes of an aligned group, in all of them.
template <int LANES>
__device__ __forceinline__ float group_sum(float x) {
  x += dpp<0xB1>(x);                              // lane ^ 1
  x += dpp<0x4E>(x);                              // lane ^ 2
  if constexpr (LANES >= 8) x += dpp<0x141>(x);   // the other four of eight, whose sums are equal
  if constexpr (LANES >= 16) x += dpp<0x140>(x);  // the other eight of sixteen
  if constexpr (LANES >= 32) x += from_lane_xor<16>(x);
  return x;
}
template <int LANES>
__device__ __forceinline__ float group_max(float x) {
  x = fmaxf(x, dpp<0xB1>(x));
  x = fmaxf(x, dpp<0x4E>(x));
  if constexpr (LANES >= 8) x = fmaxf(x, dpp<0x141>(x));
  if constexpr (LANES >= 16) x = fmaxf(x, dpp<0x140>(x));
  if constexpr (LANES >= 32) x = fmaxf(x, from_lane_xor<16>(x));
  return x;
}
// Maximum / sum over the lanes that differ in the bits from OFF on.
template <int OFF>
__device__ __forceinline__ float across_max(float x) {
  if constexpr (OFF < 64) return across_max<2 * OFF>(fmaxf(x, from_lane_xor<OFF>(x)));
  return x;
}
template <int OFF>
__device__ __forceinline__ float across_sum(float x) {
  if constexpr (OFF < 64) return across_sum<2 * OFF>(x + from_lane_xor<OFF>(x));
  return x;
}

// One step of the sum over a wave's row groups: the lane and its partner OFF away add up their
// column sums, each for one half of the 2 * KEEP columns they share; `col` is the first it keeps.
template <int KEEP, int OFF>
__device__ __forceinline__ void halve_columns(float (&o)[8], int lane, int& col) {
  const bool hi = lane & OFF;
  col += hi ? KEEP : 0;
#pragma unroll
  for (int e = 0; e < KEEP; ++e) {
    if constexpr (OFF >= 16) {  // the halves trade what the other one keeps
      const unsigned a = __float_as_uint(o[e]), b = __float_as_uint(o[e + KEEP]);
      unsigned x, y;
      if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        x = r[0], y = r[1];
      } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        x = r[0], y = r[1];
      }
      o[e] = __uint_as_float(x) + __uint_as_float(y);
    } else {
      const float mine = hi ? o[e + KEEP] : o[e], theirs = hi ? o[e] : o[e + KEEP];
      o[e] = mine + from_lane_xor<OFF>(theirs);
    }
  }
}

// Sum over the splits of a head in split order, for column d.  The partials were written by other
// workgroups of the same XCD or by an earlier launch, so they are read past the CU's own cache.  Lane s of
// 0..31 holds the maximum and the sum of split s and works its weight out once; the columns of 16 splits are
// requested together, since each batch is a trip to the L2 (a request past the last split gives 0).
template <int D>
__device__ __forceinline__ half_t merge_splits(const DecodeParams& p, int bh, int d) {
  constexpr int BATCH = 16, kDeviceScope = 16;
  const int at = threadIdx.x & 31;
  const int64_t first = (int64_t)(bh - 8 * p.whole) * p.splits;
  const auto ml = __builtin_amdgcn_make_buffer_rsrc(p.part_ml + first * 2, 0, p.splits * 8, 0x00020000);
  const auto po = __builtin_amdgcn_make_buffer_rsrc(p.part_o + first * D, 0, p.splits * D * 4, 0x00020000);
  const float m = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ml, 8 * min(at, p.splits - 1), 0, kDeviceScope));
  float l = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ml, 8 * at + 4, 0, kDeviceScope));
  float os[BATCH], osum = 0.f;
#pragma unroll
  for (int u = 0; u < BATCH; ++u)
    os[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(po, 4 * d + 4 * D * (u & 7), 4 * D * (u & 8), kDeviceScope));
  const float w = fast_exp2(m - group_max<32>(m));
  l = group_sum<32>(w * l);  // lanes past the last split: its weight, a sum of 0
  auto add = [&](int s0) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
      osum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s0 + u)) * os[u];
  };
  add(0);
  if (p.splits > BATCH) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
      os[u] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(po, 4 * d + 4 * D * (u & 7), 4 * D * (BATCH + (u & 8)), kDeviceScope));
    add(BATCH);
  }
  return (half_t)(osum / l);
}

template <int D, bool APPEND>
__global__ __launch_bounds__(256) void attn_decode_f16_kernel(DecodeParams p) {
  fetch_arguments<decltype(attn_decode_f16_kernel<D, APPEND>)>();
  constexpr int LPR = D / 8;            // lanes per cache row
  constexpr int GROUPS = 256 / LPR;         // row groups per workgroup
  constexpr int TILE = GROUPS * kDecRowsPerIt;
  constexpr int WAVES = 4;
  __shared__ float red_m[WAVES];
  __shared__ float red_l[WAVES];
  __shared__ float red_o[WAVES * D];
  __shared__ int last_flag;

  const int tid = threadIdx.x, lane = tid & 63;
  const int part = tid % LPR;
  const int grp = tid / LPR;
  // Head `bh` belongs to the XCD bh % 8, that is, to the blocks of that id % 8: first the XCD's whole heads, then
  // the splits of the others.
  const int slot = (int)(blockIdx.x >> 3), in_split = slot - p.whole;
  const bool is_whole = in_split < 0;
  const int split = is_whole ? 0 : in_split % p.splits, splits = is_whole ? 1 : p.splits;
  const int bh = (is_whole ? slot : p.whole + in_split / p.splits) * 8 + (int)(blockIdx.x & 7);
  if (bh >= p.BH) return;
  const int b = bh / p.H, h = bh % p.H;

  const half_t* K = (const half_t*)p.k + b * p.skb + h * p.skh + 8 * part;
  const half_t* V = (const half_t*)p.v + b * p.skb + h * p.skh + 8 * part;
  const int row_begin = split * p.chunk;
  const int row_end = is_whole ? p.L : min(row_begin + p.chunk, p.L);

  // One tile: kDecRowsPerIt rows of K and of V per lane group.  Rows past the end repeat the last
  // one (their scores are masked).  Every cache byte is used once: non-temporal loads keep the
  // stream from displacing itself in the caches and measurably raise the achieved HBM rate.
  half8 k[kDecRowsPerIt], v[kDecRowsPerIt];
  const int64_t step = (int64_t)GROUPS * p.skl, last = (int64_t)max(row_end - 1, 0) * p.skl;
  int64_t at = (int64_t)(row_begin + grp) * p.skl;  // the lane's first row of the next tile to request
  int64_t off[kDecRowsPerIt];
  auto place = [&](int r0) {  // tiles are placed in order
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) off[u] = r0 + grp + u * GROUPS < row_end ? at + u * step : last;
    at += kDecRowsPerIt * step;
  };
  auto load_k = [&] {
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) k[u] = __builtin_nontemporal_load((const half8*)(K + off[u]));
  };
  auto load_v = [&] {
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) v[u] = __builtin_nontemporal_load((const half8*)(V + off[u]));
  };
  // What the query needs is requested before the first tile, which is on its way while the query is
  // worked on.  The new row is handled by one lane group of the last split.
  half8 qh = {0, 0, 0, 0, 0, 0, 0, 0}, k_new = qh, v_new = qh, cs = qh, sn = qh;
  const bool owns_new_row = APPEND && grp == 0 && split == splits - 1;
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
  place(row_begin);
  load_k();
  load_v();
  __builtin_amdgcn_sched_barrier(0);
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
    m = group_sum<LPR>(m);
    l = 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (float)v_new[e];
  }

  float s[kDecRowsPerIt];
  auto scores = [&](int r0) {
#pragma unroll
    for (int u = 0; u < kDecRowsPerIt; ++u) {
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc += qf[e] * (float)k[u][e];
      acc = group_sum<LPR>(acc);
      s[u] = (r0 + grp + u * GROUPS < row_end) ? acc : -INFINITY;
    }
  };
  auto values = [&] {
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
      for (int e = 0; e < 8; ++e) o[e] += pu * (float)v[u][e];
    }
    m = m_new;
  };
  // The next tile's K is requested once the scores have used this one's, its V once the sums have: half a tile or
  // more is on its way at any time in the registers of one.  No request is under a condition that is joined again
  // before it is waited for: the wait would have to count it as not made, and so include it where it is.
  int r0 = row_begin;
  for (; r0 + TILE < row_end; r0 += TILE) {
    scores(r0);
    place(r0 + TILE);
    load_k();
    __builtin_amdgcn_sched_barrier(0);
    values();
    load_v();
    __builtin_amdgcn_sched_barrier(0);
  }
  if (r0 < row_end) {  // an append to an empty cache has no row here
    scores(r0);
    values();
  }

  // ---- merge the row groups (fixed order): within the wave by an exchange that halves the
  // columns a lane keeps at every step, so that in the end each lane holds the columns it will
  // write; then the four waves through LDS ----
  const float wave_m = across_max<LPR>(m);
  const float w = m == -INFINITY ? 0.f : fast_exp2(m - wave_m);
  l = across_sum<LPR>(l * w);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= w;
  int col = 8 * part;
  halve_columns<4, 32>(o, lane, col);
  halve_columns<2, 16>(o, lane, col);
  if constexpr (LPR <= 8) halve_columns<1, 8>(o, lane, col);
  if constexpr (LPR <= 4) o[0] += from_lane_xor<4>(o[0]);
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
    if (splits == 1) {  // nothing to merge
      ((half_t*)p.o)[(int64_t)bh * D + tid] = (half_t)(osum / lsum);
      return;
    }
    const int64_t part = (int64_t)(bh - 8 * p.whole) * splits + split;
    p.part_o[part * D + tid] = osum;
    if (tid == 0) {
      p.part_ml[part * 2 + 0] = M;
      p.part_ml[part * 2 + 1] = lsum;
    }
  }
  if (splits == 1 || !p.arrived) return;
  // The splits of a head share one XCD and so one L2: a completed store (vmcnt 0) is in that L2,
  // and relaxed device-scope atomics, which bypass the CU's own cache, are all the ordering
  // needed; no cache write-back or invalidation.
  wait_all_vmem();
  __syncthreads();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(p.arrived + bh - 8 * p.whole, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = before == splits - 1;
    if (last_flag)  // ready for the next launch
      __hip_atomic_store(p.arrived + bh - 8 * p.whole, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (last_flag && tid < D) ((half_t*)p.o)[(int64_t)bh * D + tid] = merge_splits<D>(p, bh, tid);
}

// The merge as a launch of its own, where the splits of a head may not meet in one L2.
template <int D>
__global__ __launch_bounds__(D) void attn_decode_merge_kernel(DecodeParams p) {
  fetch_arguments<decltype(attn_decode_merge_kernel<D>)>();
  const int bh = 8 * p.whole + blockIdx.x, d = threadIdx.x;
  ((half_t*)p.o)[(int64_t)bh * D + d] = merge_splits<D>(p, bh, d);
}

void launch_attn_decode_f16(const DecodeParams& p, int B, int D, bool append, hipStream_t stream) {
  const int heads = (B * p.H + 7) / 8, split_heads = B * p.H - 8 * p.whole;
  const dim3 grid(8 * (p.whole + p.splits * (heads - p.whole)));  // a head's splits on one XCD: see the kernel
  {
    LaunchScope scope(append ? "attn_decode_append_f16" : "attn_decode_f16", stream);
#define DEERS_DECODE_CASE(DD, APP) \
  if (D == DD && append == APP) hipLaunchKernelGGL((attn_decode_f16_kernel<DD, APP>), grid, dim3(256), 0, stream, p);
    DEERS_DECODE_CASE(32, false)
    DEERS_DECODE_CASE(32, true)
    DEERS_DECODE_CASE(64, false)
    DEERS_DECODE_CASE(64, true)
    DEERS_DECODE_CASE(128, false)
    DEERS_DECODE_CASE(128, true)
#undef DEERS_DECODE_CASE
  }
  if (p.splits > 1 && !p.arrived) {
    LaunchScope scope("attn_decode_merge", stream);
    if (D == 32)
      hipLaunchKernelGGL(attn_decode_merge_kernel<32>, dim3(split_heads), dim3(32), 0, stream, p);
    else if (D == 64)
      hipLaunchKernelGGL(attn_decode_merge_kernel<64>, dim3(split_heads), dim3(64), 0, stream, p);
    else
      hipLaunchKernelGGL(attn_decode_merge_kernel<128>, dim3(split_heads), dim3(128), 0, stream, p);
  }
}

}  // namespace deers
