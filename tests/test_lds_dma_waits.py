"""The wait states of the LDS DMA helpers, in the assembly that hipcc makes of them (no GPU). The
compiler's hazard pass does not look into inline asm, so each asm has to carry its own: one wait
state between a scalar write of M0 and the load, five where the load has an SGPR base."""

import importlib.util
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = ROOT / "esep-soup-kernels_amd" / "csrc"

PROBE = """
#include <hip/hip_runtime.h>
#include "attention.hpp"
// each form after a fresh M0, from an SGPR base that the VALU has just written, and from a kernel argument
__global__ void k_probe(const char* g, const char* const* table, float* out, int n) {
  __shared__ __align__(1024) char sm[8192];
  const char* base = table[threadIdx.x >> 6];
  for (int i = 0; i < n; ++i) {
    esep::lds_dma_x4_s(g + 64 * i, 16 * threadIdx.x, sm + 1024 * (i & 3));
    const uint64_t v = reinterpret_cast<uint64_t>(base + 128 * i);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t up = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    esep::lds_dma_x4_s(reinterpret_cast<const void*>(((uint64_t)up << 32) | lo), 16 * threadIdx.x,
                       sm + 4096);
    esep::lds_dma_x4(g + 16 * threadIdx.x + i, sm + 5120 + 1024 * (i & 1));
    esep::lds_dma_dword(g + 4 * threadIdx.x + i, sm + 7168 + 256 * (i & 3));
  }
  __builtin_amdgcn_s_waitcnt(esep::kWaitVm0);
  __syncthreads();
  out[threadIdx.x] = reinterpret_cast<float*>(sm)[threadIdx.x];
}
"""


def _instructions(asm):
    for line in asm.splitlines():
        text = line.split(";")[0].strip()
        if line.startswith("\t") and text and not text.startswith("."):
            yield text


def _waits(asm):
    """(load, wait states directly before it) of every LDS DMA."""
    states = 0
    for ins in _instructions(asm):
        nop = re.match(r"s_nop (\d+)", ins)
        if nop:
            states += int(nop.group(1)) + 1
            continue
        if re.match(r"(global|buffer|scratch)_load\w*lds", ins):
            yield ins, states
        states = 0


def test_every_lds_dma_waits(tmp_path):
    spec = importlib.util.spec_from_file_location("esep_build", CSRC.parent / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    src = tmp_path / "probe.hip"
    src.write_text(PROBE)
    res = subprocess.run([build.HIPCC, *build.CFLAGS, "--cuda-device-only", "-S", str(src), "-o", "-"],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    loads = list(_waits(res.stdout))
    assert len(loads) >= 4, res.stdout
    for ins, states in loads:
        assert states >= (5 if re.search(r"s\[\d+:\d+\]", ins) else 1), (ins, states)


@pytest.mark.parametrize("src", sorted(p.name for p in (*CSRC.glob("*.hip"), *CSRC.glob("*.hpp"))))
def test_every_lds_dma_goes_through_the_helpers(src):
    """The helpers' header alone issues an LDS DMA from inline asm."""
    code = "\n".join(l.split("//")[0] for l in (CSRC / src).read_text().splitlines())
    found = re.findall(r"\"[^\"]*load_lds[^\"]*\"", code)
    assert (len(found) == 3) if src == "attention.hpp" else not found, found
