"""The division of planes among workgroups where nothing has been timed
(csrc/chunk_rule.h), compiled for the host: at the shapes whose two choices were measured
it takes the faster one, it never leaves the chip emptier than the 2048-workgroup rule
and 650 workgroups both, and mixed precision keeps that rule."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eilmer4_amd", "csrc")
SOURCE = """
#include "chunk_rule.h"
extern "C" long untuned_chunks(long cols, long nk, int form)
{
    return e4::untuned_chunks(cols, nk, form == 0 ? 0.0 : form == 1 ? e4::CHUNK_TAIL_FP64 : e4::CHUNK_TAIL_EXACT);
}
"""


@pytest.fixture(scope="module")
def height(tmp_path_factory):
    d = tmp_path_factory.mktemp("chunk_rule")
    src, so = d / "c.cpp", d / "c.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(src)])
    f = C.CDLL(str(so)).untuned_chunks
    f.restype = C.c_long
    f.argtypes = [C.c_long, C.c_long, C.c_int]
    return lambda cols, nk, form=1: -(-nk // f(cols, nk, form))


@pytest.mark.parametrize("cols,nk,planes", [(256, 256, 32), (64, 128, 11), (36, 96, 5), (100, 20, 3), (14, 500, 10), (147, 170, 13),
                                            (81, 33, 4), (256, 40, 14), (380, 40, 7), (624, 12, 3), (12, 37, 1), (4, 32, 1)])
def test_measured_shapes(height, cols, nk, planes):
    assert height(cols, nk) == planes


@pytest.mark.parametrize("cols,nk,planes", [(81, 33, 4), (64, 128, 4), (112, 50, 3)])
def test_measured_shapes_reference_arithmetic(height, cols, nk, planes):
    assert height(cols, nk, 2) == planes


@pytest.mark.parametrize("cols", [1, 2, 7, 36, 81, 256, 380, 700, 768, 900, 2048, 5000])
def test_chip_is_filled(height, cols):
    for nk in (1, 2, 3, 7, 8, 33, 100, 512, 5000):
        many = -(-nk // -(-2048 // cols))
        for form in (1, 2):
            h = height(cols, nk, form)
            assert 1 <= h <= nk
            assert cols * -(-nk // h) >= min(650, cols * -(-nk // many))
        assert height(cols, nk, 0) == many
