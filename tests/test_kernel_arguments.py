"""What a kernel fetches of its arguments when it starts is counted from its own parameter list: up to where the compiler
lays the last of them, and nowhere by hand."""
import ctypes
import pathlib
import re
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "deers_amd" / "csrc"

PROGRAM = r"""
#include "common.h"
struct Odd { char c[3]; };
struct Wide { const void* p; int n; };
template <typename T>
__global__ void probe(T first, Odd odd, char c, const void* p, short s, Wide w, int i, Odd last) {
  deers::fetch_arguments<decltype(probe<T>)>();
  *(int*)p = i + last.c[0];
}
template __global__ void probe<int>(int, Odd, char, const void*, short, Wide, int, Odd);
extern "C" int all() { return deers::argument_bytes((decltype(probe<int>)*)nullptr); }
extern "C" int first() { return deers::argument_bytes((decltype(probe<int>)*)nullptr, 5); }
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_count_is_where_the_compiler_lays_the_arguments(tmp_path):
    src, lib, asm = (tmp_path / n for n in ("args.hip", "args.so", "args.s"))
    src.write_text(PROGRAM)
    flags = ["hipcc", "-O1", "-std=c++17", "--offload-arch=gfx950", "-I", str(CSRC), str(src)]
    subprocess.run(flags + ["-shared", "-fPIC", "-o", str(lib)], check=True, capture_output=True)
    subprocess.run(flags + ["-S", "--cuda-device-only", "-o", str(asm)], check=True, capture_output=True)
    laid = re.findall(r"\.offset:\s+(\d+)\s+\.size:\s+(\d+)\s+\.value_kind:\s+(by_value|global_buffer)", asm.read_text())
    ends = [int(offset) + int(size) for offset, size, _ in laid]
    assert len(ends) == 8
    counted = ctypes.CDLL(str(lib))
    assert counted.all() == ends[7] and counted.first() == ends[4]


def test_no_kernel_counts_its_arguments_by_hand():
    calls = {}
    for path in sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip")):
        text = path.read_text()
        for kernel, body in re.findall(r"__global__[^;{]*?(\w+_kernel)\([^;{]*\)\s*\{(.*?)\n\}", text, re.S):
            for which, named in re.findall(r"fetch_(?:first_)?arguments<(decltype\((\w+))?", body):
                calls[path.name, kernel] = which, named
    assert len(calls) >= 20
    for (_, kernel), (which, named) in calls.items():
        assert named == kernel, f"{kernel}: fetches the arguments of {which or 'a number of bytes'}"
