"""lds_copy16 overwrites M0, which the compiler's own copies to LDS keep their target in: a copy through the builtin
behind it has to set M0 again.  Looked at in the compiled code, without a GPU."""
import os
import subprocess

import pytest

from replisense_rfq_amd import _build

SRC = r"""
#include "common.h"
#include "mix_common.h"
__global__ void copies(const uint16_t* g, float* out, int n) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  uint16_t* const to = reinterpret_cast<uint16_t*>(smem);
  rfq::glds16(g + threadIdx.x * 8, to);
  rfqmix::lds_copy16(g + n, threadIdx.x * 16, 4096);
  rfq::glds16(g + 2 * n + threadIdx.x * 8, to);
  __syncthreads();
  out[threadIdx.x] = to[threadIdx.x] + to[threadIdx.x + 2048];
}
"""


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="needs hipcc")
def test_m0_is_set_again_behind_the_copy(tmp_path):
    src, asm = tmp_path / "copies.hip", tmp_path / "copies.s"
    src.write_text(SRC)
    subprocess.run([_build.HIPCC, *_build.MIX_FLAGS, f"-I{_build.CSRC / 'kernels'}", "--cuda-device-only", "-S", str(src),
                    "-o", str(asm)], check=True, capture_output=True)
    seen = [w for line in asm.read_text().splitlines() for w in ("s_mov_b32 m0", "global_load_lds_dwordx4") if w in line]
    assert seen == ["s_mov_b32 m0", "global_load_lds_dwordx4"] * 3
