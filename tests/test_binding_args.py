"""How the extension module converts its arguments, against a stub of the library that records what it
is given: a device pointer is an address and never the storage of the object that holds it."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

from deers_amd import rocm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ADDRESS = 0x7123_4567_8900

STUB = """
#include <stdint.h>
#include <stddef.h>
#include <string.h>
const void* seen_pointer; const void* seen_table[4]; int64_t seen_strides[4];
const char* deers_rocm_last_error(void) { return ""; }
int deers_rocm_fill(int dtype, void* p, size_t n, float value) { seen_pointer = p; return 0; }
int deers_rocm_dtoh(void* to, const void* from, size_t n) { seen_pointer = from; memset(to, 7, n); return 0; }
int deers_rocm_sum_squares_multi(int dtype, int n, const void* const* x, const int64_t* sizes, float* total, int add) {
  for (int i = 0; i < n; ++i) seen_table[i] = x[i];
  return 0;
}
int deers_rocm_rope_fwd(int dtype, const void* x, const int64_t* strides) {
  for (int i = 0; i < 4; ++i) seen_strides[i] = strides[i];
  return 0;
}
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    with open(os.path.join(ROOT, "deers_amd", "csrc", "py_calls.cpp")) as f:
        names = re.findall(r"\bX\((\w+), ", f.read())
    others = [n for n in names if n not in ("name", "fill", "dtoh", "sum_squares_multi", "rope_fwd")]
    assert len(others) > 20
    here = tmp_path_factory.mktemp("stub")
    src, lib = str(here / "stub.c"), str(here / "stub.so")
    with open(src, "w") as f:
        f.write(STUB + "".join(f"int deers_rocm_{n}(void) {{ return 0; }}\n" for n in others))
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", lib, src], check=True)
    rocm.load()
    rocm._calls.bind(lib, ctypes.c_void_p, rocm.RocmError, rocm._address)
    yield ctypes.CDLL(lib)
    rocm._calls.bind(rocm.LIB_PATH, ctypes.c_void_p, rocm.RocmError, rocm._address)


def filled(stub, pointer):
    rocm.fill_raw(np.float32, pointer, 1, 0.0)
    return ctypes.c_void_p.in_dll(stub, "seen_pointer").value or 0


class Handle(ctypes.c_void_p):
    pass


class Wrapper:
    def __init__(self, p):
        self._as_parameter_ = p


@pytest.mark.parametrize("pointer", [
    ADDRESS, ctypes.c_void_p(ADDRESS), Handle(ADDRESS), ctypes.c_uint64(ADDRESS), ctypes.c_size_t(ADDRESS),
    ctypes.cast(ADDRESS, ctypes.POINTER(ctypes.c_float)), np.int64(ADDRESS), Wrapper(ctypes.c_void_p(ADDRESS)),
    Wrapper(ADDRESS),
], ids=lambda p: type(p).__name__)
def test_a_device_pointer_is_passed_by_value(stub, pointer):
    assert filled(stub, pointer) == ADDRESS


def test_arrays_and_byref_are_their_addresses_as_ctypes_passes_them(stub):
    mapped = (ctypes.c_float * 4)()  # stands for pinned memory, which the device can reach
    assert filled(stub, mapped) == filled(stub, ctypes.byref(mapped)) == ctypes.addressof(mapped)


@pytest.mark.parametrize("pointer", [None, ctypes.c_void_p(), Handle(), Wrapper(None),
                                     ctypes.POINTER(ctypes.c_float)()], ids=lambda p: type(p).__name__)
def test_null(stub, pointer):
    filled(stub, ADDRESS)
    assert filled(stub, pointer) == 0


class Length1:  # as a tensor of one integer: it has an index and a length
    def __index__(self):
        return 5

    def __len__(self):
        return 1


@pytest.mark.parametrize("pointer", [
    np.zeros(4, np.float32), np.zeros((), np.int64), np.float32(1), b"12345678", bytearray(8), memoryview(b"12345678"),
    "text", 1.5, ctypes.c_float(1), ctypes.c_double(1), [ADDRESS], Length1(),
], ids=lambda p: type(p).__name__)
def test_what_is_no_address_is_refused(stub, pointer):
    filled(stub, ADDRESS)
    with pytest.raises(ctypes.ArgumentError):
        filled(stub, pointer)
    with pytest.raises(ctypes.ArgumentError):
        rocm.sum_squares_multi_raw(np.float32, [ADDRESS, pointer], [1, 1], ADDRESS)


def test_pointer_tables_convert_like_pointers(stub):
    rocm.sum_squares_multi_raw(np.float32, [ADDRESS, Handle(ADDRESS + 8), ctypes.c_uint64(ADDRESS + 16)], [1, 1, 1],
                               ADDRESS)
    assert list((ctypes.c_void_p * 4).in_dll(stub, "seen_table"))[:3] == [ADDRESS, ADDRESS + 8, ADDRESS + 16]


def test_a_table_that_shrinks_while_it_is_read(stub):
    class Shrink:
        @property
        def _as_parameter_(self):
            del table[1:]
            return ADDRESS
    table = [Shrink(), ADDRESS, ADDRESS]
    with pytest.raises(RuntimeError):
        rocm.sum_squares_multi_raw(np.float32, table, [1, 1, 1], ADDRESS)


@pytest.mark.parametrize("strides", [(64, 32, 8, 1), (64.0, 32.0, 8.0, 1.0), np.array([64, 32, 8, 1]),
                                     [np.float32(64), np.int32(32), 8, 1]])
def test_strides_are_what_int_takes(stub, strides):
    rocm._calls.rope_fwd(1, ADDRESS, tuple(strides), ADDRESS, ADDRESS, ADDRESS, None, 1, 1, 1, 32)
    assert list((ctypes.c_int64 * 4).in_dll(stub, "seen_strides")) == [64, 32, 8, 1]


def test_dtoh_writes_into_writable_host_buffers_only(stub):
    for out in (np.zeros(8, np.uint8), bytearray(8), (ctypes.c_uint8 * 8)()):
        rocm._calls.dtoh(out, ADDRESS, 8)
        assert bytes(out) == b"\x07" * 8
    fixed = np.zeros(8, np.uint8)
    fixed.setflags(write=False)
    for out, error in ((bytes(8), BufferError), (fixed, ValueError), (np.zeros((8, 2), np.uint8)[:, 0], ValueError),
                       (np.zeros(4, np.uint8), ValueError), (ctypes.c_void_p(ADDRESS), TypeError), (None, TypeError)):
        with pytest.raises(error):
            rocm._calls.dtoh(out, ADDRESS, 8)
    assert bytes(8) == b"\x00" * 8 and not fixed.any()
