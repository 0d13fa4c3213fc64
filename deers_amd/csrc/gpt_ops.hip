// The remaining device ops of a GPT training step around the attention module
// (src/models/gpt.rs:170-355, src/nn.rs:203-251, src/loss.rs:11-24):
//
//   index_select / index_add   token embedding and its gradient
//                              (src/storage/cpu.rs:555-660, 936-975)
//   rms_norm fwd / bwd         x * (mean(x^2) + eps)^-0.5   (src/nn.rs:244-251, weightless)
//   relu_sq fwd / bwd          relu(x)^2, the MLP activation (src/models/gpt.rs:196-197)
//   cross_entropy fwd / bwd    -mean_i log_softmax(logits)_i[target_i]  (src/loss.rs:11-24)
//
// The reference composes the last three from primitive tensor ops (4, 3 and 5 kernels
// with as many intermediate tensors); here each is one pass forward and one backward.
// All are HBM-bound.  Arithmetic is f32 whatever the storage type, rounded once.
#include "row_regs.h"

namespace deers {

namespace {

template <typename T> struct alignas(16) Vec16 { T e[16 / sizeof(T)]; };

template <typename T>
__device__ __forceinline__ Vec16<T> load16(const T* p) {
  return __builtin_bit_cast(Vec16<T>, *reinterpret_cast<const u32x4*>(p));
}
template <typename T>
__device__ __forceinline__ Vec16<T> load16_stream(const T* p) {
  return __builtin_bit_cast(Vec16<T>, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)));
}
template <typename T>
__device__ __forceinline__ void store16(const Vec16<T>& x, T* p) {
  *reinterpret_cast<u32x4*>(p) = __builtin_bit_cast(u32x4, x);
}
template <typename T>
__device__ __forceinline__ void store16_stream(const Vec16<T>& x, T* p) {
  __builtin_nontemporal_store(__builtin_bit_cast(u32x4, x), reinterpret_cast<u32x4*>(p));
}

__device__ __forceinline__ float wave_sum(float s) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  return s;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// ---- index_select (dim 0): out[i, :] = table[idx[i], :] ----
// One wavefront per output row.  An index outside [0, n_rows) writes a row of zeros and
// raises the sticky device error flag that the next synchronising call reports.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void index_select_kernel(const T* table, const int64_t* idx, T* out,
                                                           int64_t n_rows, int64_t n_idx, int width,
                                                           int* error_flag) {
  constexpr int kEpc = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= n_idx) return;
  const int64_t r = idx[i];
  const bool ok = r >= 0 && r < n_rows;
  if (!ok && lane == 0) atomicOr(error_flag, 1);
  const T* src = table + (ok ? r : 0) * width;
  T* dst = out + i * width;
  if constexpr (VEC) {
    for (int c = lane; c < width / kEpc; c += 64) {
      Vec16<T> v = load16(src + c * kEpc);
      if (!ok) v = Vec16<T>{};
      store16_stream(v, dst + c * kEpc);
    }
  } else {
    for (int c = lane; c < width; c += 64) dst[c] = ok ? src[c] : (T)0.f;
  }
}

// ---- index_add (dim 0): dst[idx[i], :] += src[i, :], in ascending i ----
// The order of additions is the reference's (src/storage/cpu.rs:954-975), so the result is the
// same bits and the same from run to run.  Destination rows are dealt to the workgroups by a hash:
// a workgroup reads the whole index vector once (it stays in L2), keeps the positions that name
// its rows in ascending order in LDS, and applies them.  With a workgroup per position instead,
// each scanning the vector to find out whether it is the first to name its row, 8192 tokens of
// 768 floats read 512 MB of indices through L2 and took 171 us; with at most 1024 workgroups the
// scan is 64 MB and the launch, 22 us, is mostly the rows' own traffic (three streams of 25 MB).
// A launch covers at most kIndexAddChunk positions (one 64-bit word of the LDS bitmap per
// thread); longer index vectors take one launch per slice, in order, which keeps the order of
// additions: a later slice adds to what the earlier ones left.
constexpr int kIndexAddChunk = 1 << 14;
constexpr int kIndexAddOwners = 1024;  // workgroups at most: four per CU, all resident
constexpr int kIndexAddBatch = 4;      // source rows in flight per column group
constexpr int kIndexAddCols = 4;       // column groups of 64 units a wave has in flight

// dst row `out` += the source rows at positions list[64 * w + b] for every bit b of hits(w),
// w = w0, w0 + 1, ..., in that order, for the columns c_first + lane, + c_step, ... of the row's
// units of EPU elements (16 bytes, or one element where rows are not whole aligned chunks).  The
// loops are uniform over the wave: `hits` may be a ballot.
template <typename T, int EPU, typename Hits>
__device__ __forceinline__ void add_rows(const T* src, T* out, const uint16_t* list, int words, int w0, int width,
                                         int c_first, int c_step, int lane, Hits hits) {
  struct alignas(sizeof(T) * EPU) Unit { T e[EPU]; };
  const int n_units = width / EPU;
  for (int base = c_first; base < n_units; base += c_step * kIndexAddCols) {
    const int c0 = base + lane;
    Unit acc[kIndexAddCols];
#pragma unroll
    for (int k = 0; k < kIndexAddCols; ++k)
      if (c0 + k * c_step < n_units) acc[k] = *(const Unit*)(out + (int64_t)(c0 + k * c_step) * EPU);
    for (int w = w0; w < words; ++w) {
      unsigned long long bits = hits(w);
      while (bits) {
        Unit x[kIndexAddBatch][kIndexAddCols];
        int n = 0;
#pragma unroll
        for (int u = 0; u < kIndexAddBatch; ++u) {
          if (!bits) break;
          const T* row = src + (int64_t)list[64 * w + __builtin_ctzll(bits)] * width;
          bits &= bits - 1;
          ++n;
#pragma unroll
          for (int k = 0; k < kIndexAddCols; ++k)
            if (c0 + k * c_step < n_units) x[u][k] = *(const Unit*)(row + (int64_t)(c0 + k * c_step) * EPU);
        }
#pragma unroll
        for (int u = 0; u < kIndexAddBatch; ++u) {
          if (u >= n) break;
#pragma unroll
          for (int k = 0; k < kIndexAddCols; ++k)
#pragma unroll
            for (int e = 0; e < EPU; ++e)  // rounded to T after each addition, as `+=` on the storage type
              acc[k].e[e] = (T)((float)acc[k].e[e] + (float)x[u][k].e[e]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kIndexAddCols; ++k)
      if (c0 + k * c_step < n_units) *(Unit*)(out + (int64_t)(c0 + k * c_step) * EPU) = acc[k];
  }
}

template <typename T, int EPU>
__global__ __launch_bounds__(256) void index_add_kernel(const T* src, const int64_t* idx, T* dst,
                                                        int64_t n_rows, int n_idx, int width,
                                                        int* error_flag) {
  extern __shared__ uint16_t list[];  // this workgroup's positions, ascending (room for n_idx)
  __shared__ unsigned long long bitmap[kIndexAddChunk / 64];
  __shared__ int wave_total[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned owner_mask = gridDim.x - 1;  // a power of two of workgroups
  const int groups = (n_idx + 63) / 64;       // at most 256
  constexpr int kInFlight = 8;
  for (int g0 = wave; g0 < groups; g0 += 4 * kInFlight) {
    int64_t r[kInFlight];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const int pos = (g0 + 4 * u) * 64 + lane;
      r[u] = pos < n_idx ? idx[pos] : -1;
    }
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const int g = g0 + 4 * u;
      if (g >= groups) break;
      const bool ok = r[u] >= 0 && r[u] < n_rows;
      const unsigned owner = ((unsigned)r[u] * 0x9E3779B1u) >> 16;
      const unsigned long long mask = __ballot(ok && (owner & owner_mask) == blockIdx.x);
      if (lane == 0) bitmap[g] = mask;
      if (blockIdx.x == 0 && !ok && g * 64 + lane < n_idx) atomicOr(error_flag, 1);
    }
  }
  __syncthreads();
  // the set bits' positions, in order: a prefix sum over the words' counts, one word per thread
  const unsigned long long mine = tid < groups ? bitmap[tid] : 0;
  const int count = __popcll(mine);
  int before = count;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int other = __shfl_up(before, off, 64);
    if (lane >= off) before += other;
  }
  if (lane == 63) wave_total[wave] = before;
  __syncthreads();
  int at = before - count, total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) at += wave_total[w];
    total += wave_total[w];
  }
  for (unsigned long long bits = mine; bits; bits &= bits - 1)
    list[at++] = (uint16_t)(tid * 64 + __builtin_ctzll(bits));
  __syncthreads();
  if (total <= 64) {
    // the usual case: the list fits a wave's lanes, the waves share out its rows
    const int64_t row = lane < total ? idx[list[lane]] : -1;
    for (int j = wave; j < total; j += 4) {
      const int64_t rj = idx[list[j]];
      const unsigned long long hits = __ballot(row == rj);
      if (hits & ((1ull << j) - 1)) continue;  // an earlier entry names this row
      add_rows<T, EPU>(src, dst + rj * width, list, 1, 0, width, 0, 64, lane, [&](int) { return hits; });
    }
  } else {
    // a row that many positions name (or an unlucky hash): every wave takes its columns of every row
    const int words = (total + 63) / 64;
    auto hits_of = [&](int w, int64_t rj) {
      const int e = 64 * w + lane;
      return __ballot(e < total && idx[list[e < total ? e : 0]] == rj);
    };
    for (int j = 0; j < total; ++j) {
      const int64_t rj = idx[list[j]];
      bool first = true;
      for (int w = 0; w <= j / 64 && first; ++w) {
        const unsigned long long hits = hits_of(w, rj);
        first = !(w == j / 64 ? hits & ((1ull << (j & 63)) - 1) : hits);
      }
      if (!first) continue;
      add_rows<T, EPU>(src, dst + rj * width, list, words, j / 64, width, wave * 64, 256, lane,
                       [&](int w) { return hits_of(w, rj); });
    }
  }
}

// ---- rms_norm: y = x * (mean(x^2) + eps)^-0.5 over the last axis ----
// One wavefront per row (rows of a transformer are 192 .. 8192 wide, a few KB): the
// second sweep over the row is served by L1/L2, so x crosses HBM once.

template <typename T, bool VEC>
__device__ __forceinline__ float row_sum_prod(const T* a, const T* b, int width, int lane) {
  constexpr int kEpc = 16 / sizeof(T);
  float s = 0.f;
  if constexpr (VEC) {
    for (int c = lane; c < width / kEpc; c += 64) {
      const Vec16<T> va = load16(a + c * kEpc), vb = load16(b + c * kEpc);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) s = fmaf((float)va.e[e], (float)vb.e[e], s);
    }
  } else {
    for (int c = lane; c < width; c += 64) s = fmaf((float)a[c], (float)b[c], s);
  }
  return wave_sum(s);
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rms_norm_fwd_kernel(const T* x, T* y, int64_t outer, int width,
                                                           float eps) {
  constexpr int kEpc = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= outer) return;
  const T* row = x + r * width;
  T* orow = y + r * width;
  const float inv = 1.0f / sqrtf(row_sum_prod<T, VEC>(row, row, width, lane) / (float)width + eps);
  if constexpr (VEC) {
    for (int c = lane; c < width / kEpc; c += 64) {
      Vec16<T> v = load16(row + c * kEpc);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) v.e[e] = (T)((float)v.e[e] * inv);
      store16(v, orow + c * kEpc);
    }
  } else {
    for (int c = lane; c < width; c += 64) orow[c] = (T)((float)row[c] * inv);
  }
}

// The forward for rows of at most 64 * RES 16-byte chunks (aligned): the row stays in the
// wave's registers between the sum of squares and the scaling.  Same bits as the general kernel.
template <typename T, int RES>
__global__ __launch_bounds__(256) void rms_norm_fwd_resident_kernel(const T* x, T* y, int64_t outer, int width,
                                                                    float eps) {
  constexpr int kEpc = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= outer) return;
  const T* row = x + r * width;
  T* orow = y + r * width;
  const int n_chunks = width / kEpc;
  Vec16<T> v[RES];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < RES; ++i) {
    const int c = lane + 64 * i;
    if (c < n_chunks) {
      v[i] = load16(row + c * kEpc);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) s = fmaf((float)v[i].e[e], (float)v[i].e[e], s);
    }
  }
  const float inv = 1.0f / sqrtf(wave_sum(s) / (float)width + eps);
#pragma unroll
  for (int i = 0; i < RES; ++i) {
    const int c = lane + 64 * i;
    if (c >= n_chunks) continue;
#pragma unroll
    for (int e = 0; e < kEpc; ++e) v[i].e[e] = (T)((float)v[i].e[e] * inv);
    store16(v[i], orow + c * kEpc);
  }
}

// dx = inv * dy - x * (inv^3 / n) * sum(dy * x), plus `addend` where one is given: the
// gradient is rounded to the storage type before the addition, as a separate add would see it
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rms_norm_bwd_kernel(const T* x, const T* dy, const T* addend, T* dx,
                                                           int64_t outer, int width, float eps) {
  constexpr int kEpc = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= outer) return;
  const T* row = x + r * width;
  const T* grow = dy + r * width;
  T* orow = dx + r * width;
  const T* arow = addend ? addend + r * width : nullptr;
  const float inv = 1.0f / sqrtf(row_sum_prod<T, VEC>(row, row, width, lane) / (float)width + eps);
  const float dot = row_sum_prod<T, VEC>(row, grow, width, lane);
  const float k = dot * inv * inv * inv / (float)width;
  if constexpr (VEC) {
    for (int c = lane; c < width / kEpc; c += 64) {
      const Vec16<T> vx = load16(row + c * kEpc), vg = load16(grow + c * kEpc);
      Vec16<T> o;
#pragma unroll
      for (int e = 0; e < kEpc; ++e) o.e[e] = (T)((float)vg.e[e] * inv - (float)vx.e[e] * k);
      if (arow) {
        const Vec16<T> va = load16(arow + c * kEpc);
#pragma unroll
        for (int e = 0; e < kEpc; ++e) o.e[e] = (T)((float)va.e[e] + (float)o.e[e]);
      }
      store16(o, orow + c * kEpc);
    }
  } else {
    for (int c = lane; c < width; c += 64) {
      const T g = (T)((float)grow[c] * inv - (float)row[c] * k);
      orow[c] = arow ? (T)((float)arow[c] + (float)g) : g;
    }
  }
}

// The same for rows of at most 64 * RES 16-byte chunks (aligned): a wave keeps its row of x
// and dy in registers, so each is read once instead of three and two times.  Sums run in
// the order of the general kernel: same bits.
template <typename T, int RES>
__global__ __launch_bounds__(256) void rms_norm_bwd_resident_kernel(const T* x, const T* dy, const T* addend,
                                                                    T* dx, int64_t outer, int width, float eps) {
  constexpr int kEpc = 16 / sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= outer) return;
  const T* row = x + r * width;
  const T* grow = dy + r * width;
  T* orow = dx + r * width;
  const T* arow = addend ? addend + r * width : nullptr;
  const int n_chunks = width / kEpc;
  Vec16<T> vx[RES], vg[RES];
#pragma unroll
  for (int i = 0; i < RES; ++i) {
    const int c = lane + 64 * i;
    if (c < n_chunks) {
      vx[i] = load16(row + c * kEpc);
      vg[i] = load16(grow + c * kEpc);
    } else {
#pragma unroll
      for (int e = 0; e < kEpc; ++e) {
        vx[i].e[e] = (T)0.f;
        vg[i].e[e] = (T)0.f;
      }
    }
  }
  float sxx = 0.f, sxg = 0.f;
#pragma unroll
  for (int i = 0; i < RES; ++i)
#pragma unroll
    for (int e = 0; e < kEpc; ++e) {
      sxx = fmaf((float)vx[i].e[e], (float)vx[i].e[e], sxx);
      sxg = fmaf((float)vx[i].e[e], (float)vg[i].e[e], sxg);
    }
  const float inv = 1.0f / sqrtf(wave_sum(sxx) / (float)width + eps);
  const float k = wave_sum(sxg) * inv * inv * inv / (float)width;
#pragma unroll
  for (int i = 0; i < RES; ++i) {
    const int c = lane + 64 * i;
    if (c >= n_chunks) continue;
    Vec16<T> o;
#pragma unroll
    for (int e = 0; e < kEpc; ++e) o.e[e] = (T)((float)vg[i].e[e] * inv - (float)vx[i].e[e] * k);
    if (arow) {
      const Vec16<T> va = load16(arow + c * kEpc);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) o.e[e] = (T)((float)va.e[e] + (float)o.e[e]);
    }
    store16(o, orow + c * kEpc);
  }
}

// ---- relu_sq: y = relu(x)^2; dx = dy * 2 * relu(x) ----
// The reference's autograd adds the two equal contributions dy * r of `r * r`
// (src/ops.rs EWiseMul backward): rounding dy * r to the storage type first and then
// doubling keeps the same bits, also where the product is subnormal in f16.
template <typename T>
__device__ __forceinline__ T relu_sq_grad(float dy, float r) {
  const float g = (float)(T)(dy * r);
  return (T)(g + g);
}
template <typename T, bool BWD>
__global__ __launch_bounds__(256) void relu_sq_kernel(const T* x, const T* dy, T* out, int64_t n) {
  constexpr int kEpc = 16 / sizeof(T);
  const int64_t n_chunks = n / kEpc;
  const int64_t stride = (int64_t)gridDim.x * 256;
  const int64_t tid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t c = tid; c < n_chunks; c += stride) {
    const Vec16<T> vx = load16_stream(x + c * kEpc);
    Vec16<T> vg, o;
    if constexpr (BWD) vg = load16_stream(dy + c * kEpc);
#pragma unroll
    for (int e = 0; e < kEpc; ++e) {
      const float r = fmaxf((float)vx.e[e], 0.f);
      if constexpr (BWD) o.e[e] = relu_sq_grad<T>((float)vg.e[e], r);
      else o.e[e] = (T)(r * r);
    }
    store16_stream(o, out + c * kEpc);
  }
  const int64_t i = n_chunks * kEpc + tid;
  if (i < n) {
    const float r = fmaxf((float)x[i], 0.f);
    if constexpr (BWD) out[i] = relu_sq_grad<T>((float)dy[i], r);
    else out[i] = (T)(r * r);
  }
}
template <typename T, bool BWD>
__global__ __launch_bounds__(256) void relu_sq_unaligned_kernel(const T* x, const T* dy, T* out,
                                                                int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float r = fmaxf((float)x[i], 0.f);
    if constexpr (BWD) out[i] = relu_sq_grad<T>((float)dy[i], r);
    else out[i] = (T)(r * r);
  }
}

// ---- cross entropy ----
// Forward: lse_i = ln sum exp(x_i) and loss_i = lse_i - x_i[target_i] per row; a second tiny
// kernel averages the per-row losses in a fixed order.  The log-probabilities are never written.
// With GRAD also dlogits[r, c] = (exp(x - lse) - [c == target]) * inv_n, the gradient of the mean
// loss for an upstream gradient of one: same expression, same bits as cross_entropy_bwd_kernel's.
// A row is held on chip by the thread group that owns it, reduced there and written from there,
// so the logits cross HBM once (row_regs.h); with and without GRAD the reduction is the same, so
// are lse and loss.  HBM-bound: [8192, 50257] f32, 1.65 GB in and 1.65 GB out.
//   A workgroup only reads until its row has arrived and only writes after that, so a CU needs two
// of them to keep both directions busy: the widest rows leave NLDS of their chunks in LDS, where
// the loads put them without passing through registers, so that the rest and the arithmetic fit
// the 64 registers two 1024-thread workgroups leave each thread: 585 us = 5.6 TB/s, where one
// workgroup of 512 threads holding 28 chunks each took 694 us = 4.7 TB/s.
template <typename T, int GROUP, int NREG, int NLDS, bool GRAD>
__global__ __launch_bounds__(kRegBlockOf(GROUP), NLDS ? 8 : 1) void cross_entropy_fwd_kernel(
    const T* logits, const int64_t* targets, float* row_lse, float* row_loss, T* dlogits, float inv_n,
    int64_t n_rows, int width, int* error_flag) {
  fetch_arguments<decltype(cross_entropy_fwd_kernel<T, GROUP, NREG, NLDS, GRAD>)>();
  __shared__ float red_m[16], red_s[16];
  extern __shared__ u32x4 parked[];  // [NLDS][GROUP]
  constexpr int kRows = kRegBlockOf(GROUP) / GROUP;
  constexpr int kEpc = 16 / sizeof(T);
  static_assert(NLDS == 0 || kRows == 1, "one row per workgroup where LDS holds a part of it");
  const int t = threadIdx.x % GROUP;
  const int64_t r = (int64_t)blockIdx.x * kRows + threadIdx.x / GROUP;
  const bool live = r < n_rows;  // whole groups only: GROUP == 64 when kRows > 1
  const T* row = logits + (live ? r : 0) * width;
  const RowGeom<T> geo(row, width);
  const int n_chunks = live ? geo.n_chunks : 0;  // a dead group's descriptors cover nothing
  // Row position of this thread's chunk 0, element 0.  Chunk u is looked at as chunk 0 of the row's
  // rest from u * GROUP chunks on (`left` elements, uniform): one register tells where all of them lie.
  const int lo0 = t * kEpc - geo.head;
  auto left = [&](int u) { return width - u * GROUP * kEpc; };
  if constexpr (NLDS > 0) {
    const uint32_t wave_lds = lds_address(parked) + (threadIdx.x & ~63) * 16;
#pragma unroll
    for (int u = 0; u < NLDS; ++u) {  // chunks past the row's end repeat its last one and are patched below
      const int chunk = min(t + (NREG + u) * GROUP, n_chunks - 1);
      async_load16_to_lds_nt(geo.base_of(row), (uint32_t)chunk * 16, wave_lds, u * GROUP * 16);
    }
  }
  u32x4 c[NREG];
#pragma unroll
  for (int u = 0; u < NREG; ++u) {
    c[u] = u32x4{0u, 0u, 0u, 0u};
    // chunks wholly before the row (slice 0 only) are not read
    if (u > 0 || lo0 + kEpc > 0) c[u] = chunk_load(slice_rsrc(geo.base_of(row), n_chunks, u * GROUP), t * 16);
  }
  const int64_t target = live ? targets[r] : 0;
  const bool ok = target >= 0 && target < width;
  const float x_target = ok ? (float)row[target] : 0.f;
#pragma unroll
  for (int u = 0; u < NREG; ++u) {
    if ((u == 0 && lo0 < 0) || lo0 + kEpc > left(u)) c[u] = patch_outside<T>(c[u], lo0, left(u), -INFINITY, u == 0);
  }
  if constexpr (NLDS > 0) wait_all_vmem();  // a thread reads only what its own wave loaded: no barrier
  auto chunk_of = [&](int u, float(&f)[kEpc]) {
    if (u < NREG) {
      keep_packed<T>(c[u < NREG ? u : 0]);
      unpack<T>(c[u < NREG ? u : 0], f);
    } else {
      u32x4 x = parked[(u - NREG) * GROUP + threadIdx.x];
      if (lo0 + kEpc > left(u)) x = patch_outside<T>(x, lo0, left(u), -INFINITY, false);
      unpack<T>(x, f);
    }
  };
  // ends a chunk's work before the next one's begins: no registers for more than one beside the row
  auto settle = [](float& x) {
    asm volatile("" : "+v"(x));
    __builtin_amdgcn_sched_barrier(0);
  };
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < NREG + NLDS; ++u) {
    float f[kEpc];
    chunk_of(u, f);
#pragma unroll
    for (int e = 0; e < kEpc; ++e) m = fmaxf(m, f[e]);
    if (NLDS > 0) settle(m);
  }
  float s = 0.f;
  if (m != -INFINITY) {
#pragma unroll
    for (int u = 0; u < NREG + NLDS; ++u) {
      float f[kEpc];
      chunk_of(u, f);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) s += __expf(f[e] - m);
      if (NLDS > 0) settle(s);
    }
  }
  group_reduce_ms<GROUP>(m, s, red_m, red_s, t);
  if (!live) return;
  const float lse = __logf(s) + m;
  if (t == 0) {
    if (!ok) atomicOr(error_flag, 1);
    row_lse[r] = lse;
    row_loss[r] = ok ? lse - x_target : 0.f;
  }
  if constexpr (GRAD) {
    T* orow = dlogits + r * width;
    // 16-byte stores need the output row at the input row's offset from a 16-byte boundary
    const bool same = same_phase(orow, row);
    const char* obase = geo.base_of(orow);
    const int hit = ok ? (int)target : INT32_MIN / 2;
#pragma unroll
    for (int u = 0; u < NREG + NLDS; ++u) {
      const int hit_u = hit - u * GROUP * kEpc;
      float f[kEpc];
      chunk_of(u, f);
#pragma unroll
      for (int e = 0; e < kEpc; ++e) {
        const float pr = __expf(f[e] - lse);
        f[e] = (pr - (hit_u == lo0 + e ? 1.0f : 0.0f)) * inv_n;
      }
      if (same && (u > 0 || lo0 >= 0) && lo0 + kEpc <= left(u))
        chunk_store(pack<T>(f), slice_rsrc(obase, n_chunks, u * GROUP), t * 16);
      else
        store_inside<T>(f, orow + u * GROUP * kEpc, lo0, left(u), u == 0);
      if (NLDS > 0) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// The same for rows that no group's registers hold: one workgroup walks the row with an online
// (max, sum) pair, and a second time for the gradient.
constexpr int kCeThreads = 512;
constexpr int kCeInFlight = 4;

template <typename T, bool GRAD>
__global__ __launch_bounds__(kCeThreads) void cross_entropy_fwd_wide_kernel(
    const T* logits, const int64_t* targets, float* row_lse, float* row_loss, T* dlogits, float inv_n,
    int width, int* error_flag) {
  __shared__ float red_m[kCeThreads / 64], red_s[kCeThreads / 64];
  __shared__ float lse_all;
  constexpr int kEpc = 16 / sizeof(T);
  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const T* row = logits + r * width;
  const int head = (int)((uintptr_t)row & 15) / (int)sizeof(T);
  const T* base = row - head;  // 16-byte aligned
  const int n_chunks = (head + width + kEpc - 1) / kEpc;
  float m = -INFINITY, s = 0.f;
  for (int c0 = tid; c0 < n_chunks; c0 += kCeThreads * kCeInFlight) {
    Vec16<T> v[kCeInFlight];
    float f[kCeInFlight][kEpc];
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < kCeInFlight; ++u) {
      const int c = c0 + u * kCeThreads;
      v[u] = Vec16<T>{};
      if (c < n_chunks) v[u] = GRAD ? load16(base + c * kEpc) : load16_stream(base + c * kEpc);
    }
#pragma unroll
    for (int u = 0; u < kCeInFlight; ++u) {
      const int lo = (c0 + u * kCeThreads) * kEpc - head;  // row position of element 0
#pragma unroll
      for (int e = 0; e < kEpc; ++e) {
        const bool in = (c0 + u * kCeThreads) < n_chunks && lo + e >= 0 && lo + e < width;
        f[u][e] = in ? (float)v[u].e[e] : -INFINITY;
        mx = fmaxf(mx, f[u][e]);
      }
    }
    if (mx > m) {
      s *= (m == -INFINITY) ? 0.f : __expf(m - mx);
      m = mx;
    }
    if (m != -INFINITY) {
#pragma unroll
      for (int u = 0; u < kCeInFlight; ++u)
#pragma unroll
        for (int e = 0; e < kEpc; ++e) s += __expf(f[u][e] - m);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
    merge_ms(m, s, m2, s2);
  }
  if ((tid & 63) == 0) {
    red_m[tid >> 6] = m;
    red_s[tid >> 6] = s;
  }
  __syncthreads();
  if (tid == 0) {
    m = red_m[0];
    s = red_s[0];
    for (int w = 1; w < kCeThreads / 64; ++w) merge_ms(m, s, red_m[w], red_s[w]);
    const float lse = __logf(s) + m;
    const int64_t t = targets[r];
    const bool ok = t >= 0 && t < width;
    if (!ok) atomicOr(error_flag, 1);
    row_lse[r] = lse;
    row_loss[r] = ok ? lse - (float)row[t] : 0.f;
    lse_all = lse;
  }
  if constexpr (GRAD) {
    __syncthreads();
    const float lse = lse_all;
    const int64_t t = targets[r];
    T* obase = dlogits + r * width - head;  // the chunk grid of the input row
    const bool same = same_phase(dlogits + r * width, row);
    for (int c = tid; c < n_chunks; c += kCeThreads) {
      const Vec16<T> v = load16(base + c * kEpc);
      const int lo = c * kEpc - head;  // row position of element 0
      Vec16<T> o;
#pragma unroll
      for (int e = 0; e < kEpc; ++e) {
        const float pr = __expf((float)v.e[e] - lse);
        o.e[e] = (T)((pr - (t == lo + e ? 1.0f : 0.0f)) * inv_n);
      }
      if (same && lo >= 0 && lo + kEpc <= width) {
        store16_stream(o, obase + c * kEpc);
      } else {  // an edge chunk shares its 16 bytes with the neighbouring row
#pragma unroll
        for (int e = 0; e < kEpc; ++e)
          if (lo + e >= 0 && lo + e < width) obase[c * kEpc + e] = o.e[e];
      }
    }
  }
}

// x *= *factor, skipped where the factor is one (the gradient of a loss that is the root of
// the graph): every block reads the factor and leaves.
template <typename T>
__global__ __launch_bounds__(256) void scale_by_device_scalar_kernel(T* x, int64_t n, const float* factor) {
  const float f = *factor;
  if (f == 1.0f) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    x[i] = (T)((float)x[i] * f);
}

// loss = scale * sum(row_loss), additions in a fixed order.  One workgroup: 8 loads in flight on
// each of 1024 threads make 8192 rows one round trip (8.6 -> 4.5 us against 256 threads with one).
constexpr int kMeanThreads = 1024, kMeanInFlight = 8;

__global__ __launch_bounds__(kMeanThreads) void mean_rows_kernel(const float* row_loss, int64_t n, float scale,
                                                                 float* loss) {
  __shared__ float red[kMeanThreads / 64];
  float s = 0.f;
  for (int64_t i0 = threadIdx.x; i0 < n; i0 += kMeanThreads * kMeanInFlight) {
    float x[kMeanInFlight];
#pragma unroll
    for (int u = 0; u < kMeanInFlight; ++u) {
      const int64_t i = i0 + u * kMeanThreads;
      x[u] = i < n ? row_loss[i] : 0.f;
    }
    s += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kMeanThreads / 64; ++w) total += red[w];
    *loss = total * scale;
  }
}

// Backward: dlogits[i, c] = (exp(x[i, c] - lse_i) - [c == target_i]) * upstream / N, one
// streaming pass over the flat [N * V] array in aligned 16-byte chunks (a chunk may
// straddle two rows).  `upstream` is the gradient of the scalar loss, in device memory.
constexpr int kCeSlab = 1024;  // 16-byte chunks per block

template <typename T>
__global__ __launch_bounds__(256) void cross_entropy_bwd_kernel(
    const T* logits, const int64_t* targets, const float* row_lse, const float* upstream, T* dlogits,
    int64_t n_rows, int width, float inv_n) {
  constexpr int kEpc = 16 / sizeof(T);
  const int64_t total = n_rows * width;
  // flat elements before the first 16-byte boundary, then whole chunks, then the tail
  const int lead = (int)(((16 - ((uintptr_t)logits & 15)) & 15) / sizeof(T));
  const float g = (upstream ? *upstream : 1.0f) * inv_n;
  auto element = [&](int64_t flat, float x) -> float {
    const int64_t r = flat / width;
    const int c = (int)(flat - r * width);
    const float p = __expf(x - row_lse[r]);
    return (p - (targets[r] == c ? 1.0f : 0.0f)) * g;
  };
  const int64_t n_chunks = total > lead ? (total - lead) / kEpc : 0;
  const int64_t tid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  // each block owns one contiguous slab of kCeSlab chunks (16 KB per array): with a read
  // and a write stream, neighbouring blocks on neighbouring addresses move more bytes per
  // second than a grid-stride sweep
  const int64_t slab0 = (int64_t)blockIdx.x * kCeSlab;
  const int64_t slab1 = slab0 + kCeSlab < n_chunks ? slab0 + kCeSlab : n_chunks;
  for (int64_t c = slab0 + threadIdx.x; c < slab1; c += 256) {
    const int64_t flat0 = lead + c * kEpc;
    const Vec16<T> vx = load16_stream(logits + flat0);
    // one division per chunk; the elements after a row boundary step to the next row
    int64_t r = flat0 / width;
    int col = (int)(flat0 - r * width);
    float lse = row_lse[r];
    int64_t t = targets[r];
    Vec16<T> o;
#pragma unroll
    for (int e = 0; e < kEpc; ++e) {
      if (col == width) {
        col = 0;
        ++r;
        lse = row_lse[r];
        t = targets[r];
      }
      const float p = __expf((float)vx.e[e] - lse);
      o.e[e] = (T)((p - (t == col ? 1.0f : 0.0f)) * g);
      ++col;
    }
    store16_stream(o, dlogits + flat0);
  }
  // edge elements: fewer than 2 chunks' worth, by the first threads
  const int64_t n_edge = total - n_chunks * kEpc;
  if (tid < n_edge) {
    const int64_t flat = tid < lead ? tid : n_chunks * kEpc + tid;
    dlogits[flat] = (T)element(flat, (float)logits[flat]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void cross_entropy_bwd_unaligned_kernel(
    const T* logits, const int64_t* targets, const float* row_lse, const float* upstream, T* dlogits,
    int64_t n_rows, int width, float inv_n) {
  const int64_t total = n_rows * width;
  const float g = (upstream ? *upstream : 1.0f) * inv_n;
  for (int64_t flat = (int64_t)blockIdx.x * 256 + threadIdx.x; flat < total;
       flat += (int64_t)gridDim.x * 256) {
    const int64_t r = flat / width;
    const int c = (int)(flat - r * width);
    const float p = __expf((float)logits[flat] - row_lse[r]);
    dlogits[flat] = (T)((p - (targets[r] == c ? 1.0f : 0.0f)) * g);
  }
}

// ---- argmax over the last axis: the greedy sampling step, kept on the device so that a
// generation loop never waits for the host ----
// One workgroup per row; ties go to the lowest index; NaNs are never selected.
// 1024 threads: a 50257-wide row is then two rounds of four 16-byte loads per thread (with
// 256 threads it was six dependent rounds, 14.6 us for 32 rows).
constexpr int kArgmaxThreads = 1024;
template <typename T>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_rows_kernel(const T* x, int64_t* out, int width) {
  __shared__ float red_v[kArgmaxThreads / 64];
  __shared__ int red_i[kArgmaxThreads / 64];
  constexpr int kEpc = 16 / sizeof(T);
  constexpr int kInFlight = 4;
  const T* row = x + (int64_t)blockIdx.x * width;
  // 16-byte chunks counted from the 16-byte boundary at or before the row start (rows
  // start at any element), the two edge chunks masked; several chunks in flight per
  // thread: a row of 50257 logits is otherwise a chain of dependent round trips
  const int head = (int)((uintptr_t)row & 15) / (int)sizeof(T);
  const T* base = row - head;
  const int n_chunks = (head + width + kEpc - 1) / kEpc;
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  for (int c0 = threadIdx.x; c0 < n_chunks; c0 += kArgmaxThreads * kInFlight) {
    Vec16<T> v[kInFlight];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      v[u] = Vec16<T>{};
      if (c0 + kArgmaxThreads * u < n_chunks) v[u] = load16_stream(base + (c0 + kArgmaxThreads * u) * kEpc);
    }
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const int lo = (c0 + kArgmaxThreads * u) * kEpc - head;  // row position of element 0 of the chunk
#pragma unroll
      for (int e = 0; e < kEpc; ++e) {
        const int c = lo + e;
        const float f = (float)v[u].e[e];
        // positions ascend within a thread, so a strict comparison keeps the lowest index
        if (c >= 0 && c < width && c0 + kArgmaxThreads * u < n_chunks && f > best) {
          best = f;
          best_i = c;
        }
      }
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float v2 = __shfl_xor(best, off, 64);
    const int i2 = __shfl_xor(best_i, off, 64);
    if (v2 > best || (v2 == best && i2 < best_i)) {
      best = v2;
      best_i = i2;
    }
  }
  if ((threadIdx.x & 63) == 0) {
    red_v[threadIdx.x >> 6] = best;
    red_i[threadIdx.x >> 6] = best_i;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kArgmaxThreads / 64; ++w)
      if (red_v[w] > best || (red_v[w] == best && red_i[w] < best_i)) {
        best = red_v[w];
        best_i = red_i[w];
      }
    out[blockIdx.x] = best_i == 0x7fffffff ? 0 : best_i;  // a row of NaNs / -inf picks 0
  }
}

unsigned stream_grid(int64_t work_items) {
  const int64_t blocks = (work_items + 255) / 256;
  const int64_t cap = 256 * 16;
  return (unsigned)(blocks < 1 ? 1 : (blocks < cap ? blocks : cap));
}

}  // namespace

template <typename T>
static void index_select_t(const T* table, const int64_t* idx, T* out, int64_t n_rows, int64_t n_idx,
                           int width, int* flag, hipStream_t stream) {
  const bool vec = aligned16(table) && aligned16(out) && (width * sizeof(T)) % 16 == 0;
  const dim3 grid((unsigned)((n_idx + 3) / 4));
  if (vec)
    hipLaunchKernelGGL((index_select_kernel<T, true>), grid, dim3(256), 0, stream, table, idx, out,
                       n_rows, n_idx, width, flag);
  else
    hipLaunchKernelGGL((index_select_kernel<T, false>), grid, dim3(256), 0, stream, table, idx, out,
                       n_rows, n_idx, width, flag);
}

void launch_index_select(int dtype_f16, const void* table, const int64_t* idx, void* out,
                         int64_t n_rows, int64_t n_idx, int width, int* flag, hipStream_t stream) {
  LaunchScope scope("index_select", stream);
  if (dtype_f16)
    index_select_t((const half_t*)table, idx, (half_t*)out, n_rows, n_idx, width, flag, stream);
  else
    index_select_t((const float*)table, idx, (float*)out, n_rows, n_idx, width, flag, stream);
}

template <typename T>
static void index_add_t(const T* src, const int64_t* idx, T* dst, int64_t n_rows, int64_t n_idx, int width,
                        int* flag, hipStream_t stream) {
  constexpr int kEpc = 16 / sizeof(T);
  const bool vec = aligned16(src) && aligned16(dst) && width % kEpc == 0;
  for (int64_t first = 0; first < n_idx; first += kIndexAddChunk) {
    const int n = (int)(n_idx - first < kIndexAddChunk ? n_idx - first : kIndexAddChunk);
    unsigned owners = 1;
    while (owners < (unsigned)n && owners < kIndexAddOwners) owners *= 2;
    const size_t lds = (size_t)n * sizeof(uint16_t);
    if (vec)
      hipLaunchKernelGGL((index_add_kernel<T, kEpc>), dim3(owners), dim3(256), lds, stream, src + first * width,
                         idx + first, dst, n_rows, n, width, flag);
    else
      hipLaunchKernelGGL((index_add_kernel<T, 1>), dim3(owners), dim3(256), lds, stream, src + first * width,
                         idx + first, dst, n_rows, n, width, flag);
  }
}

void launch_index_add(int dtype_f16, const void* src, const int64_t* idx, void* dst, int64_t n_rows,
                      int64_t n_idx, int width, int* flag, hipStream_t stream) {
  LaunchScope scope("index_add", stream);
  if (dtype_f16)
    index_add_t((const half_t*)src, idx, (half_t*)dst, n_rows, n_idx, width, flag, stream);
  else
    index_add_t((const float*)src, idx, (float*)dst, n_rows, n_idx, width, flag, stream);
}

template <typename T>
static void rms_norm_t(const T* x, const T* dy, const T* addend, T* out, int64_t outer, int width, float eps,
                       bool bwd, hipStream_t stream) {
  const bool vec = aligned16(x) && aligned16(out) && (!bwd || aligned16(dy)) && aligned16(addend) &&
                   (width * sizeof(T)) % 16 == 0;
  const dim3 grid((unsigned)((outer + 3) / 4));
  constexpr int kResident = 4;  // 16-byte chunks per lane the resident backward holds of x and of dy
  if (bwd && vec && width / (int)(16 / sizeof(T)) <= 64 * kResident) {
    hipLaunchKernelGGL((rms_norm_bwd_resident_kernel<T, kResident>), grid, dim3(256), 0, stream, x, dy, addend,
                       out, outer, width, eps);
  } else if (bwd) {
    if (vec)
      hipLaunchKernelGGL((rms_norm_bwd_kernel<T, true>), grid, dim3(256), 0, stream, x, dy, addend, out,
                         outer, width, eps);
    else
      hipLaunchKernelGGL((rms_norm_bwd_kernel<T, false>), grid, dim3(256), 0, stream, x, dy, addend, out,
                         outer, width, eps);
  } else if (vec && width / (int)(16 / sizeof(T)) <= 64 * kResident) {
    hipLaunchKernelGGL((rms_norm_fwd_resident_kernel<T, kResident>), grid, dim3(256), 0, stream, x, out, outer,
                       width, eps);
  } else {
    if (vec)
      hipLaunchKernelGGL((rms_norm_fwd_kernel<T, true>), grid, dim3(256), 0, stream, x, out, outer,
                         width, eps);
    else
      hipLaunchKernelGGL((rms_norm_fwd_kernel<T, false>), grid, dim3(256), 0, stream, x, out, outer,
                         width, eps);
  }
}

void launch_rms_norm(int dtype_f16, const void* x, const void* dy, const void* addend, void* out, int64_t outer,
                     int width, float eps, int bwd, hipStream_t stream) {
  LaunchScope scope(bwd ? "rms_norm_bwd" : "rms_norm_fwd", stream);
  if (dtype_f16)
    rms_norm_t((const half_t*)x, (const half_t*)dy, (const half_t*)addend, (half_t*)out, outer, width, eps,
               bwd != 0, stream);
  else
    rms_norm_t((const float*)x, (const float*)dy, (const float*)addend, (float*)out, outer, width, eps,
               bwd != 0, stream);
}

template <typename T, bool BWD>
static void relu_sq_t(const T* x, const T* dy, T* out, int64_t n, hipStream_t stream) {
  const bool vec = aligned16(x) && aligned16(out) && (!BWD || aligned16(dy));
  if (vec)
    hipLaunchKernelGGL((relu_sq_kernel<T, BWD>), dim3(stream_grid(n / (16 / sizeof(T)) + 16)),
                       dim3(256), 0, stream, x, dy, out, n);
  else
    hipLaunchKernelGGL((relu_sq_unaligned_kernel<T, BWD>), dim3(stream_grid(n)), dim3(256), 0, stream,
                       x, dy, out, n);
}

void launch_relu_sq(int dtype_f16, const void* x, const void* dy, void* out, int64_t n, int bwd,
                    hipStream_t stream) {
  LaunchScope scope(bwd ? "relu_sq_bwd" : "relu_sq_fwd", stream);
  if (dtype_f16) {
    if (bwd) relu_sq_t<half_t, true>((const half_t*)x, (const half_t*)dy, (half_t*)out, n, stream);
    else relu_sq_t<half_t, false>((const half_t*)x, nullptr, (half_t*)out, n, stream);
  } else {
    if (bwd) relu_sq_t<float, true>((const float*)x, (const float*)dy, (float*)out, n, stream);
    else relu_sq_t<float, false>((const float*)x, nullptr, (float*)out, n, stream);
  }
}

void launch_argmax_rows(int dtype_f16, const void* x, int64_t* out, int64_t outer, int width,
                        hipStream_t stream) {
  LaunchScope scope("argmax_rows", stream);
  if (dtype_f16)
    hipLaunchKernelGGL(argmax_rows_kernel<half_t>, dim3((unsigned)outer), dim3(kArgmaxThreads), 0, stream,
                       (const half_t*)x, out, width);
  else
    hipLaunchKernelGGL(argmax_rows_kernel<float>, dim3((unsigned)outer), dim3(kArgmaxThreads), 0, stream,
                       (const float*)x, out, width);
}

// The narrowest group that holds a row on chip: few lanes without work, and as many workgroups
// per CU as the row's size allows.
template <typename T, int GROUP, int NREG, int NLDS, bool GRAD>
static void cross_entropy_fwd_go(const T* x, const int64_t* targets, float* row_lse, float* row_loss, T* dx,
                                 int64_t n_rows, int width, int* flag, hipStream_t stream) {
  constexpr int kBlock = kRegBlockOf(GROUP), kRows = kBlock / GROUP, kLds = NLDS * GROUP * 16;
  const auto kernel = cross_entropy_fwd_kernel<T, GROUP, NREG, NLDS, GRAD>;
  if constexpr (kLds > 0) {
    static bool attr_set = false;  // launches are serialised by the caller
    if (!attr_set) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr_set = true;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)((n_rows + kRows - 1) / kRows)), dim3(kBlock), kLds, stream, x, targets,
                     row_lse, row_loss, dx, (float)(1.0 / (double)n_rows), n_rows, width, flag);
}

template <typename T, bool GRAD>
static void cross_entropy_fwd_t(const T* x, const int64_t* targets, float* row_lse, float* row_loss, T* dx,
                                int64_t n_rows, int width, int* flag, hipStream_t stream) {
  const int64_t n = worst_chunks<T>(x, width);
#define DEERS_CE_TIER(GROUP, NREG, NLDS)                                                                          \
  if (n <= GROUP * (NREG + NLDS))                                                                                 \
    return cross_entropy_fwd_go<T, GROUP, NREG, NLDS, GRAD>(x, targets, row_lse, row_loss, dx, n_rows, width, flag, \
                                                            stream);
  DEERS_CE_TIER(64, 1, 0)
  DEERS_CE_TIER(64, 4, 0)
  DEERS_CE_TIER(256, 4, 0)
  DEERS_CE_TIER(256, 8, 0)
  DEERS_CE_TIER(1024, 4, 0)
  if constexpr (sizeof(T) == 4) {
    DEERS_CE_TIER(1024, 6, 2)
    DEERS_CE_TIER(1024, 9, 4)
    DEERS_CE_TIER(1024, 10, 4)
  } else {
    DEERS_CE_TIER(1024, 8, 0)
  }
#undef DEERS_CE_TIER
  hipLaunchKernelGGL((cross_entropy_fwd_wide_kernel<T, GRAD>), dim3((unsigned)n_rows), dim3(kCeThreads), 0, stream,
                     x, targets, row_lse, row_loss, dx, (float)(1.0 / (double)n_rows), width, flag);
}

void launch_cross_entropy_fwd(int dtype_f16, const void* logits, const int64_t* targets, float* row_lse,
                              float* row_loss, float* loss, void* dlogits, int64_t n_rows, int width,
                              int* flag, hipStream_t stream) {
  LaunchScope scope(dlogits ? "cross_entropy_fwd_grad" : "cross_entropy_fwd", stream);
  auto go = [&](auto* x, auto* dx) {
    if (dx) cross_entropy_fwd_t<std::decay_t<decltype(*dx)>, true>(x, targets, row_lse, row_loss, dx, n_rows, width, flag, stream);
    else cross_entropy_fwd_t<std::decay_t<decltype(*dx)>, false>(x, targets, row_lse, row_loss, dx, n_rows, width, flag, stream);
  };
  if (dtype_f16) go((const half_t*)logits, (half_t*)dlogits);
  else go((const float*)logits, (float*)dlogits);
  hipLaunchKernelGGL(mean_rows_kernel, dim3(1), dim3(kMeanThreads), 0, stream, row_loss, n_rows,
                     (float)(1.0 / (double)n_rows), loss);
}

void launch_scale_by_device_scalar(int dtype_f16, void* x, int64_t n, const float* factor, hipStream_t stream) {
  LaunchScope scope("scale_by_scalar", stream);
  if (dtype_f16)
    hipLaunchKernelGGL(scale_by_device_scalar_kernel<half_t>, dim3(stream_grid(n)), dim3(256), 0, stream,
                       (half_t*)x, n, factor);
  else
    hipLaunchKernelGGL(scale_by_device_scalar_kernel<float>, dim3(stream_grid(n)), dim3(256), 0, stream,
                       (float*)x, n, factor);
}

void launch_cross_entropy_bwd(int dtype_f16, const void* logits, const int64_t* targets,
                              const float* row_lse, const float* upstream, void* dlogits,
                              int64_t n_rows, int width, hipStream_t stream) {
  LaunchScope scope("cross_entropy_bwd", stream);
  const float inv_n = (float)(1.0 / (double)n_rows);
  const int64_t total = n_rows * width;
  const bool same_phase = (((uintptr_t)logits ^ (uintptr_t)dlogits) & 15) == 0;
  if (dtype_f16) {
    if (same_phase)
      hipLaunchKernelGGL(cross_entropy_bwd_kernel<half_t>, dim3((unsigned)(total / 8 / kCeSlab + 1)), dim3(256),
                         0, stream, (const half_t*)logits, targets, row_lse, upstream,
                         (half_t*)dlogits, n_rows, width, inv_n);
    else
      hipLaunchKernelGGL(cross_entropy_bwd_unaligned_kernel<half_t>, dim3(stream_grid(total)),
                         dim3(256), 0, stream, (const half_t*)logits, targets, row_lse, upstream,
                         (half_t*)dlogits, n_rows, width, inv_n);
  } else {
    if (same_phase)
      hipLaunchKernelGGL(cross_entropy_bwd_kernel<float>, dim3((unsigned)(total / 4 / kCeSlab + 1)), dim3(256),
                         0, stream, (const float*)logits, targets, row_lse, upstream, (float*)dlogits,
                         n_rows, width, inv_n);
    else
      hipLaunchKernelGGL(cross_entropy_bwd_unaligned_kernel<float>, dim3(stream_grid(total)), dim3(256),
                         0, stream, (const float*)logits, targets, row_lse, upstream, (float*)dlogits,
                         n_rows, width, inv_n);
  }
}

}  // namespace deers
