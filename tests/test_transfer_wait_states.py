"""Transfers issued from assembly keep the distance the hardware asks for (CPU only: hipcc cross-compiles without a GPU).

A vector memory instruction may read a scalar register five wait states after a vector instruction wrote it at the earliest.  The
compiler inserts none in front of an assembly block, and it brings spilled scalars back with vector instructions."""
import os
import re
import shutil
import subprocess

import pytest

from neuralattentionsearch_amd import build as nats_build

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = r"""
#include "nats_prefill.h"
__global__ void k(const void* p, int n, int a, int b) {
  extern __shared__ unsigned char sm[];
  const nats::RowBuffer rows(p, n);
  const uint32_t at = nats::lds_address(sm);
  rows.to_lds<16>(at, threadIdx.x * 16, a);
  rows.to_lds<4>(at, threadIdx.x * 4, a);
  rows.to_lds_pair(at, threadIdx.x * 16, threadIdx.x * 32, a);
  rows.to_lds_quad(at, threadIdx.x * 16, threadIdx.x * 32, threadIdx.x * 48, threadIdx.x * 64, a, b);
  nats::wait_transfers();
}
"""


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="no hipcc")
def test_five_wait_states_in_front_of_the_first_transfer(tmp_path):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, *nats_build.HIPCC_FLAGS, "-I", nats_build.INCLUDE, "-I", nats_build.CSRC, "--cuda-device-only", "-S", str(src),
                    "-o", str(out)], check=True, stderr=subprocess.DEVNULL)
    blocks = [b for b in re.findall(r";;?#ASMSTART\n(.*?);;?#ASMEND", out.read_text(), re.S) if "buffer_load" in b]
    assert len(blocks) == 4
    for block in blocks:
        lines = [line.strip() for line in block.strip().splitlines()]
        first = next(i for i, line in enumerate(lines) if line.startswith("buffer_load"))
        states = sum(1 + (int(line.split()[1]) if line.startswith("s_nop") else 0) for line in lines[:first])
        assert states >= 5, block
