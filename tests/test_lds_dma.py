"""The global -> LDS loads of lds_dma.hpp read M0, which a scalar instruction
writes just before: the hardware wants one wait state between the two, and the
compiler adds none around inline assembly.  A kernel with loads at several LDS
addresses is compiled for gfx950 here, and its assembly must hold that wait
state before every such load.
"""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SRC = """
#include <hip/hip_runtime.h>
#include "lds_dma.hpp"
using namespace cai4;
__global__ void k(const void *p, uint32_t n, uint32_t *o, uint32_t s) {
  __shared__ uint32_t st[4096];
  const uint32_t at = (uint32_t)(uintptr_t)(const lds_void *)st;
  const rsrc_t r = rsrc(p, n);
  for (uint32_t i = 0; i < 4; ++i) {
    lds_dma<16>(r, at + i * 4096, threadIdx.x * 16, s * i);
    lds_dma<4>(r, at + i * 4096 + 1024, threadIdx.x * 4, s * i);
  }
  dma_wait_barrier<0>();
  o[threadIdx.x] = st[threadIdx.x * 4];
}
"""


def wait_states_after_m0(asm):
    """For every load with an LDS destination: the wait states since M0 was written."""
    out, since = [], None
    for line in asm.splitlines():
        op = line.split(";")[0].strip()
        if not op or op.startswith(".") or op.endswith(":"):
            continue
        if op.startswith("buffer_load") and op.split()[-1] == "lds":
            out.append(since)
        if re.match(r"s_\w+ m0\b", op):
            since = 0
        elif since is not None:
            nop = re.match(r"s_nop (\d+)", op)
            since += int(nop.group(1)) + 1 if nop else 1
    return out


def test_a_wait_state_between_m0_and_every_lds_load(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    src, asm = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SRC)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--cuda-device-only", "-S",
                    "-I", os.path.join(ROOT, "cascadia_amd", "csrc"), "-o", str(asm), str(src)],
                   check=True, capture_output=True, timeout=300)
    waits = wait_states_after_m0(asm.read_text())
    assert len(waits) == 8 and all(w is None or w >= 1 for w in waits), waits
    assert any(w is not None for w in waits), "M0 is not written: nothing was checked"
