"""The loads into LDS are written as inline assembly, in which the compiler places no wait states: the text that it emits
for them must hold them itself.  After a scalar write of M0 a load with an LDS destination needs one wait state, and after
a vector instruction's write of a scalar register a load that reads the register needs five.  Compiled here, not run."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zk-deepseek_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = """
#include "lds_dma.h"
extern "C" __global__ void plain(const char *p) { zk::lds_dma16(p + threadIdx.x * 16, threadIdx.y * 1024); }
extern "C" __global__ void based(const char *p)
{
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    zk::lds_dma16_uniform((uint64_t)p + w * 4096, (threadIdx.x & 63) * 16, (unsigned)w * 1024);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no compiler")
def test_loads_into_lds_wait_for_their_scalar_registers(tmp_path):
    src, out = tmp_path / "dma.hip", tmp_path / "dma.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-I", CSRC, str(src), "-o", str(out)],
                   check=True, capture_output=True)
    blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", out.read_text(), flags=re.S)
    blocks = [[l.strip() for l in b.splitlines() if l.strip()] for b in blocks]
    loads = [b for b in blocks if any(l.startswith("global_load_lds") for l in b)]
    assert len(loads) == 2

    def waits(lines):               # wait states that these instructions give
        return sum(int(l.split()[1]) + 1 if l.startswith("s_nop") else 1 for l in lines)

    for b in loads:
        at = next(i for i, l in enumerate(b) if l.startswith("global_load_lds"))
        m0 = max(i for i, l in enumerate(b[:at]) if re.match(r"s_mov_b32 m0,", l))
        assert waits(b[m0 + 1:at]) >= 1, b
        if not b[at].rstrip().endswith("off"):          # the address comes from a scalar register pair
            assert waits(b[:at]) >= 5, b
