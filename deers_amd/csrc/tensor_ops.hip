// Element-wise helpers the fused attention op needs from its storage backend:
// gradient accumulation (`existing + grad`, src/backprop.rs:101-112 through
// BinaryOp Add, src/storage.rs:231-236), compaction of a strided view
// (copy_compact, src/storage.rs:305; CPU form src/storage/cpu.rs:1063-1102),
// the constant fill behind ones_like/zeros_like (src/backprop.rs:54) and unary
// negation (src/ops.rs:100-127).  All are bandwidth-bound one-pass kernels.
#include "common.h"

namespace deers {

namespace {

template <typename T>
__device__ __forceinline__ float to_f32(T v) { return (float)v; }

template <typename T>
__global__ __launch_bounds__(256) void fill_kernel(T* dst, size_t n, float value) {
  const T v = (T)value;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    dst[i] = v;
}

// f16 adds go through f32 and round once, like `half`'s software `+`.
template <typename T>
__global__ __launch_bounds__(256) void add_kernel(const T* a, const T* b, T* out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    out[i] = (T)(to_f32(a[i]) + to_f32(b[i]));
}

template <typename T>
__global__ __launch_bounds__(256) void neg_kernel(const T* a, T* out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    out[i] = (T)(-to_f32(a[i]));
}

// A strided copy: up to six dimensions, outermost first, each with its extent and the
// element (or 16-byte chunk) stride on either side.
template <typename I>
struct CopyView {
  I shape[6];
  I src[6];
  I dst[6];
  int ndim;
};

// dst viewed through v.dst <- src viewed through v.src, `n` units of E in all.  E is uint4
// where both sides are whole aligned 16-byte chunks, else the element; I is 32-bit where every
// offset fits.  The index arithmetic (a division per dimension) is what an element-wise 64-bit
// form was bound by: 32 prompts of 512 x 12 heads x 64 halves into a KV cache, 25 MB each way,
// took 79 us = 0.6 TB/s; one division chain per 16 bytes, in 32 bits, over dimensions the host
// has merged: 10.8 us = 4.7 TB/s.
template <typename E, typename I>
__global__ __launch_bounds__(256) void copy_view_kernel(const E* src, E* dst, CopyView<I> v, I n) {
  fetch_arguments<decltype(copy_view_kernel<E, I>)>();
  for (I i = (I)blockIdx.x * 256 + threadIdx.x; i < n; i += (I)gridDim.x * 256) {
    I rem = i, so = 0, dof = 0;
    for (int d = v.ndim - 1; d > 0; --d) {
      const I q = rem / v.shape[d], idx = rem - q * v.shape[d];
      so += idx * v.src[d];
      dof += idx * v.dst[d];
      rem = q;
    }
    dst[dof + rem * v.dst[0]] = src[so + rem * v.src[0]];
  }
}

inline unsigned grid_for(size_t n) {
  const size_t blocks = (n + 255) / 256;
  return (unsigned)(blocks < 1 ? 1 : (blocks > 16384 ? 16384 : blocks));
}

}  // namespace

void launch_fill(int dtype_f16, void* dst, size_t n, float value, hipStream_t stream) {
  if (dtype_f16)
    hipLaunchKernelGGL(fill_kernel<half_t>, dim3(grid_for(n)), dim3(256), 0, stream, (half_t*)dst, n, value);
  else
    hipLaunchKernelGGL(fill_kernel<float>, dim3(grid_for(n)), dim3(256), 0, stream, (float*)dst, n, value);
}

void launch_add(int dtype_f16, const void* a, const void* b, void* out, size_t n,
                hipStream_t stream) {
  if (dtype_f16)
    hipLaunchKernelGGL(add_kernel<half_t>, dim3(grid_for(n)), dim3(256), 0, stream,
                       (const half_t*)a, (const half_t*)b, (half_t*)out, n);
  else
    hipLaunchKernelGGL(add_kernel<float>, dim3(grid_for(n)), dim3(256), 0, stream,
                       (const float*)a, (const float*)b, (float*)out, n);
}

void launch_neg(int dtype_f16, const void* a, void* out, size_t n, hipStream_t stream) {
  if (dtype_f16)
    hipLaunchKernelGGL(neg_kernel<half_t>, dim3(grid_for(n)), dim3(256), 0, stream,
                       (const half_t*)a, (half_t*)out, n);
  else
    hipLaunchKernelGGL(neg_kernel<float>, dim3(grid_for(n)), dim3(256), 0, stream,
                       (const float*)a, (float*)out, n);
}

template <typename E, typename I>
static void copy_view_as(const void* src, void* dst, const CopyView<int64_t>& v, int64_t n, hipStream_t stream) {
  CopyView<I> u;
  u.ndim = v.ndim;
  for (int d = 0; d < v.ndim; ++d) {
    u.shape[d] = (I)v.shape[d];
    u.src[d] = (I)v.src[d];
    u.dst[d] = (I)v.dst[d];
  }
  hipLaunchKernelGGL((copy_view_kernel<E, I>), dim3(grid_for((size_t)n)), dim3(256), 0, stream, (const E*)src,
                     (E*)dst, u, (I)n);
}

// dst viewed through dst_strides <- src viewed through src_strides, same shape.
void launch_copy_view(int dtype_f16, const void* src, const int64_t* src_strides, void* dst,
                      const int64_t* dst_strides, const int64_t* shape, int ndim,
                      hipStream_t stream) {
  // extents of one vanish, neighbouring dimensions that step alike on both sides become one
  CopyView<int64_t> v;
  v.ndim = 0;
  int64_t n = 1;
  for (int d = 0; d < ndim; ++d) {
    n *= shape[d];
    if (shape[d] == 1) continue;
    const int last = v.ndim - 1;
    if (last >= 0 && v.src[last] == src_strides[d] * shape[d] && v.dst[last] == dst_strides[d] * shape[d]) {
      v.shape[last] *= shape[d];
    } else {
      v.shape[v.ndim++] = shape[d];
    }
    v.src[v.ndim - 1] = src_strides[d];
    v.dst[v.ndim - 1] = dst_strides[d];
  }
  if (n == 0) return;
  if (v.ndim == 0) {
    v.shape[0] = 1;
    v.src[0] = v.dst[0] = 1;
    v.ndim = 1;
  }
  // Whole 16-byte chunks: unit innermost strides, and every other step, the innermost extent
  // and both addresses multiples of 16 bytes.
  const int64_t per16 = dtype_f16 ? 8 : 4;
  const int in = v.ndim - 1;
  bool chunked = v.src[in] == 1 && v.dst[in] == 1 && v.shape[in] % per16 == 0 &&
                 ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
  int64_t src_span = 1, dst_span = 1;
  for (int d = 0; d <= in; ++d) {
    if (d < in) chunked = chunked && v.src[d] % per16 == 0 && v.dst[d] % per16 == 0;
    src_span += (v.shape[d] - 1) * v.src[d];
    dst_span += (v.shape[d] - 1) * v.dst[d];
  }
  int64_t span = src_span > dst_span ? src_span : dst_span;
  if (n > span) span = n;
  if (chunked) {
    for (int d = 0; d < in; ++d) {
      v.src[d] /= per16;
      v.dst[d] /= per16;
    }
    v.shape[in] /= per16;
    n /= per16;
    span /= per16;
  }
  // 32-bit indices, with room for the grid stride past the last unit
  const bool narrow = span < (int64_t(1) << 31);
  if (chunked) {
    if (narrow) copy_view_as<uint4, uint32_t>(src, dst, v, n, stream);
    else copy_view_as<uint4, int64_t>(src, dst, v, n, stream);
  } else if (dtype_f16) {
    if (narrow) copy_view_as<uint16_t, uint32_t>(src, dst, v, n, stream);
    else copy_view_as<uint16_t, int64_t>(src, dst, v, n, stream);
  } else {
    if (narrow) copy_view_as<uint32_t, uint32_t>(src, dst, v, n, stream);
    else copy_view_as<uint32_t, int64_t>(src, dst, v, n, stream);
  }
}

// dst (compact, row-major over `shape`) <- src viewed through `strides`.
void launch_copy_strided(int dtype_f16, const void* src, const int64_t* shape,
                         const int64_t* strides, int ndim, void* dst, hipStream_t stream) {
  int64_t compact[6], run = 1;
  for (int d = ndim - 1; d >= 0; --d) {
    compact[d] = run;
    run *= shape[d];
  }
  launch_copy_view(dtype_f16, src, strides, dst, compact, shape, ndim, stream);
}

}  // namespace deers
