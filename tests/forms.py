"""Which form of the attention kernels a launch takes: the library's own rules, and its test hook."""
import contextlib
import ctypes

import numpy as np

from deers_amd import rocm


def takes_32_rows(direction, dtype, heads, T, D):
    """Whether this launch takes the 32-row form (for the f32 backward: whether it computes S and dP twice)."""
    i64 = ctypes.c_int64
    if direction == "bwd" and dtype == np.float32:
        return rocm.load()["_ZN5deers18attn_bwd_f32_headsEllll"](i64(heads), i64(T), i64(D), i64(2304 << 20)) == 0
    rule = rocm.load()[f"_ZN5deers24attn_{direction}_f{16 if dtype == np.float16 else 32}_split_takesElll"]
    rule.restype = ctypes.c_bool
    return rule(i64(heads), i64(T), i64(D))


def scores_from_q(heads, T, D):
    """Whether this f16 launch, forward and backward, forms its scores from Q itself, not from Q * scale * log2(e) in f16."""
    rule = rocm.load()["_ZN5deers15attn_f16_from_qElllf"]
    rule.restype = ctypes.c_bool
    i64 = ctypes.c_int64
    return rule(i64(heads), i64(T), i64(D), ctypes.c_float(rocm.default_scale(D)))


@contextlib.contextmanager
def rows_128(on=True):
    """Launches take the 128-row kernels wherever there is one, whatever their size."""
    rocm.debug_attn_128_rows(on)
    try:
        yield
    finally:
        rocm.debug_attn_128_rows(False)
