"""The orders in which workgroups take blocks of falling length.  Those that are all resident at once: every block once,
and the CUs' totals closer together than in the order of length itself.  Heads that the XCDs cannot share out whole:
the closed form against the rule it stands for."""
import ctypes
import shutil
import subprocess

import pytest

ROOT = __file__.rsplit("/", 2)[0]

PROGRAM = r"""
#include "common.h"
extern "C" int block(int id, int grid, int cus) { return deers::paired_block(id, grid, cus); }
extern "C" int even_blocks(int n_ranks, int heads) { return deers::map_even_blocks(n_ranks, heads); }
extern "C" int even(int id, int n_ranks, int heads, int by_search) {
  int head, rank;
  const auto map = by_search ? deers::map_block_even_by_search : deers::map_block_even;
  return map(id, n_ranks, heads, &head, &rank) ? rank * heads + head : -1;
}
"""


pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")


@pytest.fixture(scope="module")
def maps(tmp_path_factory):
    tmp_path = tmp_path_factory.mktemp("order")
    src, lib = tmp_path / "order.hip", tmp_path / "order.so"
    src.write_text(PROGRAM)
    subprocess.run(["hipcc", "-shared", "-fPIC", "-O1", "-std=c++17", "--offload-arch=gfx950", "-I",
                    ROOT + "/deers_amd/csrc", str(src), "-o", str(lib)], check=True, capture_output=True)
    return ctypes.CDLL(str(lib))


def test_every_block_once_and_even_totals(maps):
    block = maps.block
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


def test_blocks_of_heads_that_the_xcds_cannot_share_out_whole(maps):
    """Rank by rank: the remaining heads' blocks go to the XCDs in turn, the whole heads stay on their XCD; a list that
    is shorter than the longest ends in ids that name no block."""
    for heads in list(range(1, 42)) + [63, 64, 65, 100, 263]:
        for n_ranks in (1, 2, 3, 5, 8, 17):
            lists, dealt = [[] for _ in range(8)], 0
            for rank in range(n_ranks):
                for head in range(heads - heads % 8, heads):
                    lists[dealt % 8].append(rank * heads + head)
                    dealt += 1
                for head in range(heads - heads % 8):
                    lists[head % 8].append(rank * heads + head)
            grid = maps.even_blocks(n_ranks, heads)
            assert grid == 8 * max(map(len, lists))
            for by_search in (0, 1):
                taken = [[maps.even(8 * i + xcd, n_ranks, heads, by_search) for i in range(grid // 8)] for xcd in range(8)]
                assert taken == [x + [-1] * (grid // 8 - len(x)) for x in lists], (heads, n_ranks)
