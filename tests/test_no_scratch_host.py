"""The face kernel of mixture blocks built from their grid holds everything in
registers.  (Its solves run in a loop over the two sides of a face; a local array
indexed by the side is put in scratch, 32 bytes a lane, without a word from the
compiler.)  Compiled here for one form; the size is the kernel descriptor's."""
import os
import re
import shutil
import subprocess

import pytest

from eilmer4_amd import build

SOURCE = """
#include "gen_kernels.h"
namespace e4 { template __global__ void gen_face_kernel<ModeFast64, 5, 0, 0>(TPArgs); }
"""


@pytest.mark.skipif(not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)), reason="no hipcc")
def test_grid_mixture_faces_have_no_scratch(tmp_path):
    src, asm = tmp_path / "g.hip", tmp_path / "g.s"
    src.write_text(SOURCE)
    subprocess.check_call([build.HIPCC] + build.COMMON + ["-ffp-contract=fast", "--cuda-device-only", "-S", "-I", build.CSRC,
                                                          "-o", str(asm), str(src)], stderr=subprocess.DEVNULL)
    sizes = re.findall(r"\.amdhsa_kernel (\S*gen_face_kernel\S*).*?private_segment_fixed_size (\d+)", asm.read_text(), re.S)
    assert sizes and all(n == "0" for _, n in sizes), sizes
