// Rows held in registers: what the row-wise kernels (log-softmax, cross-entropy) share.
#pragma once

#include "common.h"

namespace deers {

namespace {

__device__ __forceinline__ void merge_ms(float& m, float& s, float m2, float s2) {
  const float mn = fmaxf(m, m2);
  // (-inf, 0) is the neutral element; guard its exp(-inf - -inf)
  const float a = (m == -INFINITY) ? 0.f : __expf(m - mn);
  const float b = (m2 == -INFINITY) ? 0.f : __expf(m2 - mn);
  s = s * a + s2 * b;
  m = mn;
}

// GROUP threads own one row; a workgroup of kRegBlock threads holds kRegBlock / GROUP
// rows.  The row is cut into 16-byte chunks counted from the 128-byte line its first
// element lies in (rows start at any element: 50257 is odd), so that every access is a
// full-width dwordx4 and every wavefront access covers whole cache lines.  Chunks
// before the row are skipped; the chunks that straddle the row's ends hold neighbours'
// elements, which are replaced by the reduction's neutral element after the load and
// never stored.
// Thread t of the group holds chunks t, t + GROUP, ... (NREG of them, packed as loaded,
// so an f16 row takes half the registers of an f32 row).

constexpr int kRegBlockOf(int group) { return group < 256 ? 256 : group; }
template <int GROUP>
__device__ __forceinline__ void group_reduce_ms(float& m, float& s, float* red_m, float* red_s,
                                                int t) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
    merge_ms(m, s, m2, s2);
  }
  if constexpr (GROUP > 64) {
    if ((t & 63) == 0) {
      red_m[t >> 6] = m;
      red_s[t >> 6] = s;
    }
    __syncthreads();
    // every wave merges the waves' results for itself: a tree over its first lanes (a chain of
    // GROUP / 64 merges took 0.6 us of a 16-wave row and the registers of all the results)
    m = red_m[t & (GROUP / 64 - 1)];
    s = red_s[t & (GROUP / 64 - 1)];
#pragma unroll
    for (int off = GROUP / 128; off >= 1; off >>= 1) {
      const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
      merge_ms(m, s, m2, s2);
    }
  }
  // a merge is not the same bits with its operands exchanged: one lane's result for all
  m = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m)));
  s = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(s)));
}

template <int GROUP>
__device__ __forceinline__ float group_reduce_sum(float s, float* red, int t) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if constexpr (GROUP > 64) {
    if ((t & 63) == 0) red[t >> 6] = s;
    __syncthreads();
    s = red[0];
#pragma unroll
    for (int w = 1; w < GROUP / 64; ++w) s += red[w];
  }
  return s;
}

// A 16-byte chunk as loaded, and its elements as floats.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Elems { T e[16 / sizeof(T)]; };

template <typename T>
__device__ __forceinline__ void unpack(u32x4 c, float (&f)[16 / sizeof(T)]) {
  const Elems<T> x = __builtin_bit_cast(Elems<T>, c);
#pragma unroll
  for (int e = 0; e < (int)(16 / sizeof(T)); ++e) f[e] = (float)x.e[e];
}
template <typename T>
__device__ __forceinline__ u32x4 pack(const float (&f)[16 / sizeof(T)]) {
  Elems<T> x;
#pragma unroll
  for (int e = 0; e < (int)(16 / sizeof(T)); ++e) x.e[e] = (T)f[e];
  return __builtin_bit_cast(u32x4, x);
}

// Makes the compiler forget what it knows about a packed chunk, so that f16 -> f32
// conversions are redone where the values are used instead of being kept live (which
// would triple the registers an f16 row takes).
template <typename T>
__device__ __forceinline__ void keep_packed(u32x4& c) {
  if constexpr (sizeof(T) == 2) asm volatile("" : "+v"(c));
}

// Slices of a row are addressed through buffer descriptors (base and extent in SGPRs,
// advanced with scalar arithmetic) and ONE 32-bit byte offset per lane, which keeps
// address arithmetic out of the vector registers that hold the row.  The extent ends
// at the last chunk that overlaps the row: chunks past it load zeros and touch no
// memory.  aux = 2 marks the access non-temporal: every byte is used once.
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr int kAuxNt = 2;

__device__ __forceinline__ rsrc_t slice_rsrc(const char* base, int n_chunks, int first_chunk) {
  const int left = n_chunks > first_chunk ? n_chunks - first_chunk : 0;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)first_chunk * 16), 0, left * 16,
                                           0x00020000);
}
__device__ __forceinline__ u32x4 chunk_load(rsrc_t r, int byte_off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, kAuxNt));
}
__device__ __forceinline__ void chunk_store(u32x4 c, rsrc_t r, int byte_off) {
  __builtin_amdgcn_raw_buffer_store_b128(
      __builtin_bit_cast(__attribute__((__vector_size__(4 * sizeof(unsigned int)))) unsigned int, c),
      r, byte_off, 0, kAuxNt);
}

// Where a row lies relative to its chunks.  Chunk 0 starts at the 128-byte line that
// holds the row's first element, so that every wavefront access covers whole cache
// lines; `head` elements (up to a line's worth) precede the row in chunks that are
// never loaded or stored.  Operands that move with the row (the output, lsm) use the
// same head, measured back from their own row start.
template <typename T>
struct RowGeom {
  int head;      // elements between the line start and the row
  int n_chunks;  // chunks from the line start to the row's end
  __device__ __forceinline__ RowGeom(const T* row, int inner) {
    constexpr int kEpc = 16 / sizeof(T);
    head = (int)((uintptr_t)row & 127) / (int)sizeof(T);
    n_chunks = (head + inner + kEpc - 1) / kEpc;
  }
  __device__ __forceinline__ const char* base_of(const T* row) const {
    return (const char*)(row - head);
  }
};

// Replaces the elements of chunk `c` (row positions lo .. lo + EPC - 1) that lie outside
// [0, inner) by `neutral` (may_precede false: none lies before 0).
template <typename T>
__device__ __forceinline__ u32x4 patch_outside(u32x4 c, int lo, int inner, float neutral, bool may_precede = true) {
  constexpr int kEpc = 16 / sizeof(T);
  Elems<T> x = __builtin_bit_cast(Elems<T>, c);
#pragma unroll
  for (int e = 0; e < kEpc; ++e)
    if ((may_precede && lo + e < 0) || lo + e >= inner) x.e[e] = (T)neutral;
  return __builtin_bit_cast(u32x4, x);
}

// Stores the elements of an edge chunk that belong to the row, one by one.
template <typename T>
__device__ __forceinline__ void store_inside(const float (&f)[16 / sizeof(T)], T* orow, int lo,
                                             int inner, bool may_precede = true) {
#pragma unroll
  for (int e = 0; e < (int)(16 / sizeof(T)); ++e)
    if ((!may_precede || lo + e >= 0) && lo + e < inner) orow[lo + e] = (T)f[e];
}

// Chunks from a row's line start to its end, at worst over all rows.  Row r starts
// (first + r * pitch) mod 128 bytes into its line; those offsets step by gcd(pitch, 128).
template <typename T>
int64_t worst_chunks(const T* first_row, int64_t inner) {
  constexpr int kEpc = 16 / sizeof(T);
  const int64_t pitch = inner * (int64_t)sizeof(T);
  int64_t g = 128;
  while (pitch % g) g /= 2;
  const int64_t max_head_bytes = (int64_t)((uintptr_t)first_row % (uintptr_t)g) + 128 - g;
  return (max_head_bytes / (int64_t)sizeof(T) + inner + kEpc - 1) / kEpc;
}
__host__ __device__ inline bool same_phase(const void* a, const void* b) {
  return (((uintptr_t)a ^ (uintptr_t)b) & 15) == 0;
}

// 16 chunks of f32 (64 values) fill the 128 VGPRs a 1024-thread workgroup leaves each
// thread; an f16 chunk unpacks to 8 floats while it is worked on, so 8 is its limit.
template <typename T> constexpr int kMaxChunksPerThread = sizeof(T) == 4 ? 16 : 8;

}  // namespace

}  // namespace deers
