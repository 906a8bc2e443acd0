"""The index arithmetic of csrc/block_index.h, compiled for the host, over blocks up to
the largest that fit the memory: cell indices beyond 2^29 (whose byte offset is beyond
32 bits) and 2^31."""
import ctypes as C
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eilmer4_amd", "csrc")
SOURCE = """
#include "block_index.h"
extern "C" {
int reach_block(int d, int ni, int nj, int nk) { return e4::offsets_reach_block(d, ni, nj, nk); }
long row_start(int ni, int nj, int j, int k) { return e4::row_start(ni, nj, j, k); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("block_index")
    src, so = d / "b.cpp", d / "b.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(src)])
    L = C.CDLL(str(so))
    L.row_start.restype = C.c_long
    return L


@pytest.mark.parametrize("n", [(820, 820, 820), (1024, 1024, 512), (1500, 1500, 1600), (25000, 25000, 1), (2, 2 ** 30 + 5, 1),
                               (2 ** 30 + 5, 2, 1), (2, 40000, 40000), (130, 9, 5), (2, 2, 2)])
def test_rows(lib, n):
    ni, nj, nk = n
    rng = random.Random(ni)
    for j, k in [(0, 0), (nj - 1, 0), (0, nk - 1), (nj - 1, nk - 1)] + [(rng.randrange(nj), rng.randrange(nk)) for _ in range(50)]:
        assert lib.row_start(ni, nj, j, k) == (k * nj + j) * ni


@pytest.mark.parametrize("n", [(812, 812, 813), (813, 813, 813), (820, 820, 820), (23170, 23170, 1), (23171, 23170, 1),
                               (2 ** 28 - 1, 2, 1), (2 ** 28, 2, 1), (2, 2 ** 28, 1), (2, 2, 2 ** 27), (2, 2, 2 ** 27 - 1),
                               (2 ** 31 - 1, 2, 1), (128, 128, 128)])
def test_blocks_out_of_reach(lib, n):
    """The byte offset of every cell and face within its field is below 2^32 exactly where
    the rule says so."""
    ni, nj, nk = n
    dims = 2 if nk == 1 else 3
    most = max((ni + 1) * nj * nk, ni * (nj + 1) * nk, ni * nj * (nk + 1) if dims == 3 else 0)
    assert bool(lib.reach_block(dims, ni, nj, nk)) == (8 * (most - 1) < 2 ** 32)
