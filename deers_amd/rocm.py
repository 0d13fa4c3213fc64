"""Python binding of the C ABI in include/deers_rocm.h (no torch).  The calls that a training step or
a generated token consists of go through the extension module `_calls`, the others through ctypes.

This is host-side plumbing for tests and the benchmark: device buffers, copies,
timers and the three attention entry points, called exactly the way a
`Device::Rocm` storage backend in deers would call them over `extern "C"`.
There is no CPU fallback: if the HIP library is missing or no gfx950 device is
present, every call raises.
"""
from __future__ import annotations

import ctypes
import importlib
import operator
import os

import numpy as np

F16, F32 = 0, 1
_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("DEERS_ROCM_LIB") or os.path.join(_HERE, "libdeers_rocm.so")

_lib = None
_inited = False


class _NotLoaded:
    """Stands in for the extension until the first call through it."""

    def __getattr__(self, name):
        load()
        return getattr(_calls, name)


_calls = _NotLoaded()


class RocmError(RuntimeError):
    """A non-zero return code from the library (the role of deers' backend error variant)."""


_BYREF = type(ctypes.byref(ctypes.c_int()))
_INTEGER_CODES = "bBhHiIlLqQ"  # of ctypes' simple types


def _address(o) -> int:
    """The address that a pointer argument stands for, if it is no None, int or c_void_p: what ctypes passes
    for its own pointers, integers and arrays and for byref(), an object's `_as_parameter_`, or an integer
    of another type.  Everything else is refused, a numpy array or a tensor above all: its storage may be
    host memory, and its one element is no address."""
    if isinstance(o, ctypes._SimpleCData):
        if isinstance(o, ctypes.c_void_p) or o._type_ in _INTEGER_CODES:
            return o.value or 0
    elif isinstance(o, (ctypes._Pointer, ctypes.Array, _BYREF)):
        return ctypes.cast(o, ctypes.c_void_p).value or 0
    elif hasattr(o, "_as_parameter_"):
        p = o._as_parameter_
        return 0 if p is None else p if isinstance(p, int) else _address(p)
    elif hasattr(o, "__index__") and not hasattr(o, "__len__"):
        return operator.index(o)
    raise ctypes.ArgumentError(f"a pointer argument cannot be of type {type(o).__name__}")


def load() -> ctypes.CDLL:
    """Loads libdeers_rocm.so and the extension module; raises if they have not been built."""
    global _lib, _calls
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RocmError(
                f"{LIB_PATH} is missing: build it with `make -C deers_amd/csrc` "
                "(or __graft_entry__.build()); there is no fallback path")
        lib = ctypes.CDLL(LIB_PATH)
        lib.deers_rocm_last_error.restype = ctypes.c_char_p
        lib.deers_rocm_stream.restype = ctypes.c_void_p
        try:
            calls = importlib.import_module("deers_amd._calls")
        except ImportError as e:
            raise RocmError(f"the extension module deers_amd._calls is missing ({e}): build it with "
                            "`make -C deers_amd/csrc` (or __graft_entry__.build())") from e
        calls.bind(LIB_PATH, ctypes.c_void_p, RocmError, _address)
        _lib, _calls = lib, calls
    return _lib


def _check(rc: int):
    if rc != 0:
        raise RocmError(f"deers_rocm error {rc}: {load().deers_rocm_last_error().decode()}")


def available() -> bool:
    return bool(load().deers_rocm_available())


def init(ordinal: int = 0):
    global _inited
    if not _inited:
        _check(load().deers_rocm_init(ctypes.c_int(ordinal)))
        _inited = True


def sync():
    _check(load().deers_rocm_sync())


HANDOVER_STREAM_ORDER, HANDOVER_SAME_XCD = 0, 1


def handover_policy(cu_count: int, cu_mask_set: bool) -> int:
    """deers_rocm_handover_policy: the rule alone, no device needed."""
    return int(load().deers_rocm_handover_policy(ctypes.c_int(cu_count), ctypes.c_int(int(cu_mask_set))))


def handover_mode() -> int:
    """Mode in force: HANDOVER_SAME_XCD / HANDOVER_STREAM_ORDER, -1 before init."""
    return int(load().deers_rocm_handover_mode())


def set_handover_mode(mode: int):
    _check(load().deers_rocm_set_handover_mode(ctypes.c_int(mode)))


def debug_bwd_wait(spin_limit: int = 1 << 20, skip_producers: bool = False):
    """Test hook of the single-launch backward's bounded wait (see the header)."""
    _check(load().deers_rocm_debug_bwd_wait(ctypes.c_int(spin_limit), ctypes.c_int(int(skip_producers))))


def debug_attn_128_rows(on: bool):
    """Test hook: attention calls take the 128-row kernels wherever there is one (see the header)."""
    _check(load().deers_rocm_debug_attn_128_rows(ctypes.c_int(int(on))))


_CODES = {np.float16: F16, np.float32: F32}


def dtype_code(dtype) -> int:
    code = _CODES.get(dtype)
    if code is not None:
        return code
    dtype = np.dtype(dtype)
    if dtype == np.float16:
        return F16
    if dtype == np.float32:
        return F32
    raise TypeError(f"unsupported dtype {dtype}")


class DeviceBuffer:
    """An owned device allocation with a shape and dtype (compact row-major)."""

    def __init__(self, shape, dtype, zeros: bool = False):
        init()
        self.shape = tuple(int(s) for s in shape)
        self.dtype = np.dtype(dtype)
        self.nbytes = int(np.prod(self.shape)) * self.dtype.itemsize
        ptr = ctypes.c_void_p()
        fn = load().deers_rocm_alloc_zeros if zeros else load().deers_rocm_alloc
        _check(fn(ctypes.c_size_t(self.nbytes), ctypes.byref(ptr)))
        self.ptr = ptr

    @classmethod
    def from_numpy(cls, a: np.ndarray) -> "DeviceBuffer":
        a = np.ascontiguousarray(a)
        buf = cls(a.shape, a.dtype)
        _check(load().deers_rocm_htod(buf.ptr, a.ctypes.data_as(ctypes.c_void_p),
                                      ctypes.c_size_t(buf.nbytes)))
        return buf

    def numpy(self) -> np.ndarray:
        out = np.empty(self.shape, dtype=self.dtype)
        _calls.dtoh(out, self.ptr, self.nbytes)
        return out

    def free(self):
        if self.ptr is not None and self.ptr.value:
            _check(load().deers_rocm_free(self.ptr))
        self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class Timer:
    """hipEvent pair on the library stream."""

    def __init__(self):
        init()
        self.h = ctypes.c_void_p()
        _check(load().deers_rocm_timer_create(ctypes.byref(self.h)))

    def start(self):
        _check(load().deers_rocm_timer_start(self.h))

    def stop(self):
        _check(load().deers_rocm_timer_stop(self.h))

    def elapsed_ms(self) -> float:
        ms = ctypes.c_float()
        _check(load().deers_rocm_timer_elapsed_ms(self.h, ctypes.byref(ms)))
        return float(ms.value)

    def __del__(self):
        try:
            load().deers_rocm_timer_destroy(self.h)
        except Exception:
            pass


def profile_enable(on: bool = True):
    """Switch per-kernel event timing on (clears earlier records) or off."""
    init()
    _check(load().deers_rocm_profile_enable(ctypes.c_int(1 if on else 0)))


def matmul_tune(on: bool):
    _check(load().deers_rocm_matmul_tune(ctypes.c_int(1 if on else 0)))


def empty_cache():
    _check(load().deers_rocm_empty_cache())


def set_bwd_workspace_limit(nbytes: int = -1):
    """deers_rocm_set_bwd_workspace_limit: memory for the f32 backward's dS (-1: the default, 0: none)."""
    init()
    _check(load().deers_rocm_set_bwd_workspace_limit(ctypes.c_int64(nbytes)))


def profile_collect() -> dict:
    """{kernel name: (calls, total_ms)} for launches since profile_enable(True)."""
    n = ctypes.c_int()
    _check(load().deers_rocm_profile_collect(ctypes.byref(n)))
    out = {}
    for i in range(n.value):
        name, calls, ms = ctypes.c_char_p(), ctypes.c_int64(), ctypes.c_float()
        _check(load().deers_rocm_profile_row(ctypes.c_int(i), ctypes.byref(name),
                                             ctypes.byref(calls), ctypes.byref(ms)))
        out[name.value.decode()] = (int(calls.value), float(ms.value))
    return out


def attn_fwd_raw(dtype, q, k, v, o, lse, B, H, T, D, scale, q_strides=None, k_strides=None,
                 v_strides=None, o_strides=None):
    """deers_rocm_attn_fwd on raw device pointers (DeviceBuffer.ptr)."""
    _calls.attn_fwd(dtype_code(dtype), q, q_strides, k, k_strides, v, v_strides, o, o_strides, lse, B, H, T, D, scale)


def attn_bwd_raw(dtype, q, k, v, o, lse, do, dq, dk, dv, B, H, T, D, scale, strides=None):
    """deers_rocm_attn_bwd on raw device pointers; `strides` maps tensor name -> 4 strides."""
    g = (strides or {}).get
    _calls.attn_bwd(dtype_code(dtype), q, g("q"), k, g("k"), v, g("v"), o, g("o"), lse, do, g("do"), dq, g("dq"), dk,
                    g("dk"), dv, g("dv"), B, H, T, D, scale)


def attn_decode_raw(dtype, q, k_cache, v_cache, o, B, H, L, D, scale, kv_strides=None):
    _calls.attn_decode(dtype_code(dtype), q, k_cache, v_cache, kv_strides, o, B, H, L, D, scale)


def attn_decode_noalloc_raw(dtype, q, k_cache, v_cache, o, B, H, L, D, scale, kv_strides=None):
    """deers_rocm_attn_decode_noalloc: attn_decode with the split partials in static device memory."""
    ks = None if kv_strides is None else (ctypes.c_int64 * 3)(*[int(x) for x in kv_strides])
    _check(load().deers_rocm_attn_decode_noalloc(
        ctypes.c_int(dtype_code(dtype)), q, k_cache, v_cache, ks, o, ctypes.c_int64(B),
        ctypes.c_int64(H), ctypes.c_int64(L), ctypes.c_int64(D), ctypes.c_float(scale)))


def attn_decode_append_raw(dtype, q, k, v, in_strides, cos_row, sin_row, k_cache, v_cache, cache_strides,
                           o, pos, capacity, B, H, D, scale):
    """deers_rocm_attn_decode_append: rotate q, k at `pos`, append k, v as cache row pos, attend over [0,pos]."""
    _calls.attn_decode_append(dtype_code(dtype), q, k, v, in_strides, cos_row, sin_row, k_cache, v_cache, cache_strides,
                              o, pos, capacity, B, H, D, scale)


def fill_raw(dtype, dst, n, value):
    _calls.fill(dtype_code(dtype), dst, n, value)


def add_raw(dtype, a, b, out, n):
    _check(load().deers_rocm_add(ctypes.c_int(dtype_code(dtype)), a, b, out, ctypes.c_size_t(n)))


def neg_raw(dtype, a, out, n):
    _check(load().deers_rocm_neg(ctypes.c_int(dtype_code(dtype)), a, out, ctypes.c_size_t(n)))


def copy_compact_raw(dtype, src, shape, strides, dst):
    """dst (compact over `shape`) <- src read through element `strides`."""
    nd = len(shape)
    sh = (ctypes.c_int64 * nd)(*[int(x) for x in shape])
    st = (ctypes.c_int64 * nd)(*[int(x) for x in strides])
    _check(load().deers_rocm_copy_compact(ctypes.c_int(dtype_code(dtype)), src, sh, st,
                                          ctypes.c_int(nd), dst))


def log_softmax_fwd_raw(dtype, x, out, outer, inner):
    _check(load().deers_rocm_log_softmax_fwd(ctypes.c_int(dtype_code(dtype)), x, out,
                                             ctypes.c_int64(outer), ctypes.c_int64(inner)))


def log_softmax_bwd_raw(dtype, grad, lsm, out, outer, inner):
    _check(load().deers_rocm_log_softmax_bwd(ctypes.c_int(dtype_code(dtype)), grad, lsm, out,
                                             ctypes.c_int64(outer), ctypes.c_int64(inner)))


def index_select_raw(dtype, table, indices, out, n_rows, n_indices, width):
    _calls.index_select(dtype_code(dtype), table, indices, out, n_rows, n_indices, width)


def index_add_raw(dtype, src, indices, dst, n_rows, n_indices, width):
    _calls.index_add(dtype_code(dtype), src, indices, dst, n_rows, n_indices, width)


def rms_norm_fwd_raw(dtype, x, y, outer, inner, eps):
    _calls.rms_norm_fwd(dtype_code(dtype), x, y, outer, inner, eps)


def rms_norm_bwd_raw(dtype, x, dy, dx, outer, inner, eps):
    _calls.rms_norm_bwd(dtype_code(dtype), x, dy, dx, outer, inner, eps)


def rms_norm_bwd_add_raw(dtype, x, dy, addend, dx, outer, inner, eps):
    _calls.rms_norm_bwd_add(dtype_code(dtype), x, dy, addend, dx, outer, inner, eps)


def relu_sq_fwd_raw(dtype, x, y, n):
    _calls.relu_sq_fwd(dtype_code(dtype), x, y, n)


def relu_sq_bwd_raw(dtype, x, dy, dx, n):
    _calls.relu_sq_bwd(dtype_code(dtype), x, dy, dx, n)


def argmax_rows_raw(dtype, x, out, outer, inner):
    _calls.argmax_rows(dtype_code(dtype), x, out, outer, inner)


def cross_entropy_fwd_raw(dtype, logits, targets, row_lse, loss, n_rows, n_classes):
    _calls.cross_entropy_fwd(dtype_code(dtype), logits, targets, row_lse, loss, n_rows, n_classes)


def cross_entropy_fwd_grad_raw(dtype, logits, targets, row_lse, loss, dlogits, n_rows, n_classes):
    _calls.cross_entropy_fwd_grad(dtype_code(dtype), logits, targets, row_lse, loss, dlogits, n_rows, n_classes)


def scale_by_scalar_raw(dtype, x, n, factor):
    _calls.scale_by_scalar(dtype_code(dtype), x, n, factor)


def cross_entropy_bwd_raw(dtype, logits, targets, row_lse, upstream, dlogits, n_rows, n_classes):
    _calls.cross_entropy_bwd(dtype_code(dtype), logits, targets, row_lse, upstream, dlogits, n_rows, n_classes)


# op codes of deers_rocm_unary / deers_rocm_binary / deers_rocm_reduce (include/deers_rocm.h)
UNARY_OPS = {"neg": 0, "exp": 1, "log": 2, "sin": 3, "cos": 4, "tanh": 5, "relu": 6,
             "relu_backward": 7, "scalar_add": 8, "scalar_mul": 9, "scalar_div": 10, "powf": 11}
BINARY_OPS = {"add": 0, "sub": 1, "mul": 2, "div": 3, "pow": 4, "eq": 5}
REDUCE_OPS = {"sum": 0, "max": 1}
I64 = 2


def _i64_array(values):
    if values is None:
        return None
    return (ctypes.c_int64 * len(values))(*[int(x) for x in values])


def unary_raw(dtype, op, x, shape, strides, param, out):
    """out (compact over `shape`) = op(x read through element `strides`; None = compact)."""
    _check(load().deers_rocm_unary(ctypes.c_int(dtype_code(dtype)), ctypes.c_int(UNARY_OPS[op]), x,
                                   ctypes.c_int(len(shape)), _i64_array(shape), _i64_array(strides),
                                   ctypes.c_double(param), out))


def binary_raw(dtype, op, a, a_strides, b, b_strides, shape, out):
    _check(load().deers_rocm_binary(ctypes.c_int(dtype_code(dtype)), ctypes.c_int(BINARY_OPS[op]), a,
                                    _i64_array(a_strides), b, _i64_array(b_strides),
                                    ctypes.c_int(len(shape)), _i64_array(shape), out))


def reduce_raw(dtype, op, x, out, outer, reduce_size):
    _check(load().deers_rocm_reduce(ctypes.c_int(dtype_code(dtype)), ctypes.c_int(REDUCE_OPS[op]), x, out,
                                    ctypes.c_int64(outer), ctypes.c_int64(reduce_size)))


def log_sum_exp_raw(dtype, x, out, outer, reduce_size):
    _check(load().deers_rocm_log_sum_exp(ctypes.c_int(dtype_code(dtype)), x, out, ctypes.c_int64(outer),
                                         ctypes.c_int64(reduce_size)))


def gather_raw(dtype, src, indices, out, left, src_dim, index_len, right):
    code = I64 if np.dtype(dtype) == np.int64 else dtype_code(dtype)
    _check(load().deers_rocm_gather(ctypes.c_int(code), src, indices, out, ctypes.c_int64(left),
                                    ctypes.c_int64(src_dim), ctypes.c_int64(index_len),
                                    ctypes.c_int64(right)))


def scatter_add_raw(dtype, src, indices, dst, left, dst_dim, index_len, right):
    _check(load().deers_rocm_scatter_add(ctypes.c_int(dtype_code(dtype)), src, indices, dst,
                                         ctypes.c_int64(left), ctypes.c_int64(dst_dim),
                                         ctypes.c_int64(index_len), ctypes.c_int64(right)))


def adamw_step_raw(dtype, w, grad, m, v, n, lr, beta1, beta2, eps, weight_decay, step,
                   grad_scale=1.0):
    _check(load().deers_rocm_adamw_step(
        ctypes.c_int(dtype_code(dtype)), w, grad, m, v, ctypes.c_int64(n), ctypes.c_double(lr),
        ctypes.c_double(beta1), ctypes.c_double(beta2), ctypes.c_double(eps),
        ctypes.c_double(weight_decay), ctypes.c_int64(step), ctypes.c_double(grad_scale)))


def sum_squares_raw(dtype, x, n, total, accumulate=False):
    _check(load().deers_rocm_sum_squares(ctypes.c_int(dtype_code(dtype)), x, ctypes.c_int64(n),
                                         total, ctypes.c_int(1 if accumulate else 0)))


def adamw_step_multi_raw(dtype, w, grad, m, v, sizes, lr, beta1, beta2, eps, weight_decay, step,
                         grad_scale=1.0):
    n = len(sizes)
    if not n == len(w) == len(grad) == len(m) == len(v):
        raise ValueError("as many weights, gradients and moments as sizes are needed")
    _calls.adamw_step_multi(dtype_code(dtype), n, w, grad, m, v, sizes, lr, beta1, beta2, eps, weight_decay, step,
                            grad_scale)


def sum_squares_multi_raw(dtype, x, sizes, total, accumulate=False):
    n = len(sizes)
    if n != len(x):
        raise ValueError("as many tensors as sizes are needed")
    _calls.sum_squares_multi(dtype_code(dtype), n, x, sizes, total, 1 if accumulate else 0)


def scale_raw(dtype, x, n, scale):
    _check(load().deers_rocm_scale(ctypes.c_int(dtype_code(dtype)), x, ctypes.c_int64(n),
                                   ctypes.c_double(scale)))


def matmul_raw(dtype, a, a_strides, b, b_strides, c, batch, m, n, k):
    """deers_rocm_matmul: c[batch,m,n] = a @ b; strides are (row, col, batch) in elements."""
    _calls.matmul(dtype_code(dtype), a, *a_strides[:3], b, *b_strides[:3], c, batch, m, n, k)


def matmul_acc_raw(dtype, a, a_strides, b, b_strides, c, batch, m, n, k):
    """deers_rocm_matmul_acc: c[batch,m,n] += a @ b; strides are (row, col, batch) in elements."""
    _calls.matmul_acc(dtype_code(dtype), a, *a_strides[:3], b, *b_strides[:3], c, batch, m, n, k)


def matmul_add_raw(dtype, a, a_strides, b, b_strides, addend, c, batch, m, n, k):
    """deers_rocm_matmul_add: c[batch,m,n] = a @ b + addend; strides are (row, col, batch) in elements."""
    _calls.matmul_add(dtype_code(dtype), a, *a_strides[:3], b, *b_strides[:3], addend, c, batch, m, n, k)


LINEAR_PROLOGUES = {"plain": 0, "rms_norm": 1, "relu_sq": 2}
LINEAR_W_PACKED = -32  # DEERS_ROCM_LINEAR_W_PACKED: pass as ldw for a [n/32][k][32] weight


def decode_linear_raw(dtype, prologue, eps, x, ldx, w, ldw, y, accumulate, m, n, k):
    """deers_rocm_decode_linear: y[m,n] (+)= f(x)[m,k] @ w[k,n], m <= 32, f one of LINEAR_PROLOGUES."""
    _calls.decode_linear(dtype_code(dtype), LINEAR_PROLOGUES[prologue], eps, x, ldx, w, ldw, y, 1 if accumulate else 0, m,
                         n, k)


def decode_linear_hint_raw(next_w_packed, n, k):
    """deers_rocm_decode_linear_hint: the packed weight of the product after the next one (None clears)."""
    _calls.decode_linear_hint(next_w_packed, n, k)


def decode_qkv_raw(dtype, q, k, v, in_strides, cos_row, sin_row, q_out, k_cache, v_cache, cache_strides,
                   pos, capacity, B, H, D):
    """deers_rocm_decode_qkv: rotate q, k at `pos`; q -> q_out [B,H,D]; k, v -> row pos of the caches."""
    _calls.decode_qkv(dtype_code(dtype), q, k, v, in_strides, cos_row, sin_row, q_out, k_cache, v_cache, cache_strides,
                      pos, capacity, B, H, D)


def rope_fwd_raw(dtype, x, cos, sin, y, B, T, H, D, x_strides=None, y_strides=None):
    """deers_rocm_rope_fwd: x logical [B,T,H,D] -> y [B,H,T,D] (compact unless y_strides)."""
    _calls.rope_fwd(dtype_code(dtype), x, x_strides, cos, sin, y, y_strides, B, T, H, D)


def copy_view_raw(dtype, src, src_strides, dst, dst_strides, shape):
    nd = len(shape)
    if not nd == len(src_strides) == len(dst_strides):
        raise ValueError("as many strides as dimensions are needed")
    _calls.copy_view(dtype_code(dtype), src, src_strides, dst, dst_strides, shape, nd)


def rope_bwd_raw(dtype, dy, cos, sin, dx, B, T, H, D, dy_strides=None):
    """deers_rocm_rope_bwd: dy logical [B,H,T,D] -> dx compact [B,T,H,D]."""
    _calls.rope_bwd(dtype_code(dtype), dy, dy_strides, cos, sin, dx, B, T, H, D)


def default_scale(D: int) -> float:
    """1/sqrt(D) in double, narrowed to f32 (src/models/gpt.rs:139, src/storage.rs:115-117)."""
    return float(np.float32(1.0 / np.sqrt(float(D))))


# ---- numpy-in / numpy-out conveniences (copy to the device, run, copy back) ----

def attn_fwd(q: np.ndarray, k: np.ndarray, v: np.ndarray, scale: float | None = None):
    """Returns (o, lse) for compact [B,H,T,D] numpy inputs of one dtype (f16 or f32)."""
    B, H, T, D = q.shape
    scale = default_scale(D) if scale is None else scale
    dq_, dk_, dv_ = (DeviceBuffer.from_numpy(a) for a in (q, k, v))
    o = DeviceBuffer(q.shape, q.dtype)
    lse = DeviceBuffer((B, H, T), np.float32)
    attn_fwd_raw(q.dtype, dq_.ptr, dk_.ptr, dv_.ptr, o.ptr, lse.ptr, B, H, T, D, scale)
    return o.numpy(), lse.numpy()


def attn_fwd_composed_raw(dtype, q, k, v, mask, o, lse, s, p, B, H, T, D, scale):
    """The reference's own op chain for the attention core (src/models/gpt.rs:139-144,
    softmax of src/tensor.rs:456-458) on the device, one storage kernel per tensor op:
    matmul, scalar_mul, add of the [B,1,T,T] mask broadcast over the heads, log_sum_exp,
    sub of the [B,H,T,1] statistic broadcast over the keys, exp, matmul.  What a
    Device::Rocm backend executes where the fused op does not apply (any head width).
    `s`, `p`: two [B,H,T,T] scratch buffers of `dtype`; `lse`: [B,H,T] of `dtype`."""
    BH, shape = B * H, (B, H, T, T)
    matmul_raw(dtype, q, (D, 1, T * D), k, (1, D, T * D), s, BH, T, T, D)            # q @ k^T
    unary_raw(dtype, "scalar_mul", s, shape, None, scale, p)                          # * scale
    binary_raw(dtype, "add", p, None, mask, [T * T, 0, T, 1], shape, s)               # + mask
    log_sum_exp_raw(dtype, s, lse, BH * T, T)
    binary_raw(dtype, "sub", s, None, lse, [H * T, T, 1, 0], shape, p)                # - lse
    unary_raw(dtype, "exp", p, shape, None, 0.0, s)
    matmul_raw(dtype, s, (T, 1, T * T), v, (D, 1, T * D), o, BH, T, D, T)             # @ v


def causal_mask_host(B: int, T: int, dtype) -> np.ndarray:
    """Additive mask [B,1,T,T]: -inf above the diagonal, as src/nn/functional.rs:12-55 builds it
    on the host before every forward."""
    m = np.where(np.triu(np.ones((T, T), bool), 1), -np.inf, 0.0).astype(dtype)
    return np.ascontiguousarray(np.broadcast_to(m, (B, 1, T, T)))


def attn_fwd_composed(q: np.ndarray, k: np.ndarray, v: np.ndarray, scale: float | None = None):
    """Returns (o, lse) computed by the unfused chain; compact [B,H,T,D] inputs of one dtype."""
    B, H, T, D = q.shape
    scale = default_scale(D) if scale is None else scale
    bq, bk, bv = (DeviceBuffer.from_numpy(a) for a in (q, k, v))
    mask = DeviceBuffer.from_numpy(causal_mask_host(B, T, q.dtype))
    o = DeviceBuffer(q.shape, q.dtype)
    lse = DeviceBuffer((B, H, T), q.dtype)
    s, p = DeviceBuffer((B, H, T, T), q.dtype), DeviceBuffer((B, H, T, T), q.dtype)
    attn_fwd_composed_raw(q.dtype, bq.ptr, bk.ptr, bv.ptr, mask.ptr, o.ptr, lse.ptr, s.ptr, p.ptr,
                          B, H, T, D, scale)
    return o.numpy(), lse.numpy()


def attn_fwd_bwd(q, k, v, do, scale: float | None = None):
    """Returns (o, lse, dq, dk, dv): forward then backward through the C ABI."""
    B, H, T, D = q.shape
    scale = default_scale(D) if scale is None else scale
    bq, bk, bv, bdo = (DeviceBuffer.from_numpy(a) for a in (q, k, v, do))
    o = DeviceBuffer(q.shape, q.dtype)
    lse = DeviceBuffer((B, H, T), np.float32)
    gq, gk, gv = (DeviceBuffer(q.shape, q.dtype) for _ in range(3))
    attn_fwd_raw(q.dtype, bq.ptr, bk.ptr, bv.ptr, o.ptr, lse.ptr, B, H, T, D, scale)
    attn_bwd_raw(q.dtype, bq.ptr, bk.ptr, bv.ptr, o.ptr, lse.ptr, bdo.ptr, gq.ptr, gk.ptr, gv.ptr,
                 B, H, T, D, scale)
    return o.numpy(), lse.numpy(), gq.numpy(), gk.numpy(), gv.numpy()


def attn_decode(q: np.ndarray, k_cache: np.ndarray, v_cache: np.ndarray,
                scale: float | None = None, length: int | None = None):
    """q [B,H,D], caches [B,H,Lcap,D] (f16); attends to the first `length` cache rows."""
    B, H, D = q.shape
    Lcap = k_cache.shape[2]
    L = Lcap if length is None else length
    scale = default_scale(D) if scale is None else scale
    bq, bk, bv = (DeviceBuffer.from_numpy(a) for a in (q, k_cache, v_cache))
    o = DeviceBuffer((B, H, D), q.dtype)
    attn_decode_raw(q.dtype, bq.ptr, bk.ptr, bv.ptr, o.ptr, B, H, L, D, scale,
                    kv_strides=(H * Lcap * D, Lcap * D, D))
    return o.numpy()
