"""The order in which workgroups that are all resident at once take blocks of falling length: every block once, and the
CUs' totals closer together than in the order of length itself."""
import ctypes
import shutil
import subprocess

import pytest

ROOT = __file__.rsplit("/", 2)[0]

PROGRAM = r"""
#include "common.h"
extern "C" int block(int id, int grid, int cus) { return deers::paired_block(id, grid, cus); }
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_every_block_once_and_even_totals(tmp_path):
    src, lib = tmp_path / "order.hip", tmp_path / "order.so"
    src.write_text(PROGRAM)
    subprocess.run(["hipcc", "-shared", "-fPIC", "-O1", "-std=c++17", "--offload-arch=gfx950", "-I",
                    ROOT + "/deers_amd/csrc", str(src), "-o", str(lib)], check=True, capture_output=True)
    block = ctypes.CDLL(str(lib)).block
    for cus in (32, 5):
        for n in range(cus + 1, 4 * cus + 1):
            taken = [block(8 * i + 3, 8 * n, cus) for i in range(n)]
            assert all(t % 8 == 3 for t in taken) and sorted(t // 8 for t in taken) == list(range(n))
            totals, plain = [0] * cus, [0] * cus
            for i, t in enumerate(taken):  # block i of an XCD runs on CU i % cus; lengths fall from n to 1
                totals[i % cus] += n - t // 8
                plain[i % cus] += n - i
            assert max(totals) <= max(plain)
            if n <= 2 * cus:  # nothing better than the longest alone, or a pair of the others
                assert max(totals) <= max(n, 2 * (n - cus) + 1)
