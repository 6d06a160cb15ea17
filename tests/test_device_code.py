"""What the compiler makes of the kernels' memory accesses, read from the gfx950 assembly of a few instantiations."""

import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vkgrad_amd", "csrc")
SOURCE = """
#include "gemm_dma_kernel.h"
#include "gemm_kernel.h"
namespace mg {
template __global__ void gemm_kernel<%s, D_BF16, 64, 64, 64, 2, 2, true, false>(const GemmParams);
}
"""


@pytest.mark.parametrize("layout", ["L_NN", "L_NT", "L_TN"])
def test_loads_at_any_alignment_are_global(tmp_path, layout):
    """A flat load counts as an LDS access too: a wait for fragments would wait for the K-block just asked for.  Whole K-blocks
    are loaded at a scalar base and 32-bit lane offsets, with no 64-bit address a piece to add up in every K-block."""
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE % layout)
    subprocess.run([os.environ.get("HIPCC", "hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-munsafe-fp-atomics",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "-I", CSRC,
                    "-I", os.path.join(CSRC, "..", "..", "include"), "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    asm = out.read_text()
    assert "global_load_dwordx4" in asm and "v_mfma" in asm
    assert "flat_load" not in asm and "flat_store" not in asm
    assert re.search(r"global_load_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\]", asm)
