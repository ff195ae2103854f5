"""CPU: the assembly of the DPP updates (magma_amd/csrc/dpp_fma.h).  A DPP
operand needs two wait states after the VALU instruction that writes it, and the
compiler does not look for them inside inline assembly: it may put a copy of the
operand right before any statement, so every statement with a DPP instruction
has to begin with the wait."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "magma_amd", "csrc")

SOURCE = """
#include "dpp_fma.h"
using namespace magma_amd;
template <class T>
__device__ void rows(T *p, const T *x)
{
    T a[32];
    for (int k = 0; k < 32; ++k) a[k] = p[64 * k + threadIdx.x];
    const T x0 = -x[threadIdx.x], x1 = -x[64 + threadIdx.x], l = x[128 + threadIdx.x];
    fmac_row<0, 32>(a, x0, x1, l);
    fmac_row<3, 17>(a, x0, x1, a[0]);
    fmac_row<16, 32>(a, x0, x1, a[1]);
    fmac_row<31, 32>(a, x0, x1, a[2]);
    for (int k = 0; k < 32; ++k) p[64 * k + threadIdx.x] = a[k];
}
__global__ void f64(double *p, const double *x) { rows(p, x); }
__global__ void f32(float *p, const float *x) { rows(p, x); }
"""


def test_every_statement_waits_before_its_dpp_operands(tmp_path):
    hipcc = shutil.which("hipcc", path="/opt/rocm/bin" + os.pathsep + os.environ.get("PATH", ""))
    if hipcc is None:
        pytest.skip("no hipcc")
    # inline DPP instructions stand in one file
    for f in sorted(os.listdir(CSRC)):
        if f.endswith((".h", ".hip")) and f != "dpp_fma.h":
            with open(os.path.join(CSRC, f)) as src:
                assert not re.search(r'"[^"\n]*(_dpp |row_newbcast|quad_perm)', src.read()), f
    (tmp_path / "rows.hip").write_text(SOURCE)
    subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-I" + CSRC,
                    "-I" + os.path.join(ROOT, "include"), "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    str(tmp_path / "rows.hip"), "-o", str(tmp_path / "rows.s")], check=True, capture_output=True)
    blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", (tmp_path / "rows.s").read_text(), re.S)
    blocks = [[line.strip() for line in b.splitlines() if line.strip()] for b in blocks]
    blocks = [b for b in blocks if any("_dpp" in line for line in b)]
    assert sum("_dpp" in line for b in blocks for line in b) == 2 * (32 + 14 + 16 + 1)
    for b in blocks:
        wait = re.match(r"s_nop (\d+)", b[0])
        assert wait and int(wait.group(1)) >= 1, b
        # nothing but the updates after it, none writing an operand of a later one
        for line in b[1:]:
            assert re.match(r"v_fmac_f(32|64)_dpp ", line), line
        written = [line.split()[1].rstrip(",") for line in b[1:]]
        read = {r.rstrip(",") for line in b[1:] for r in line.split()[2:4]}
        assert not read & set(written), b
