"""The rotation block of the real-rotation passes writes some of its registers before it has
read the others: no two of its operands may be given the same register, also where the compiler
knows that they hold the same number."""
import re
import subprocess

import pytest

from qandle_amd._engine import jit
from qandle_amd.csrc import build

KERNEL = """#include <hip/hip_runtime.h>
%s
extern "C" __global__ void k(float2 *p, float t, int f) {
  float2 %s;
  rot_pairs%d(%s, t, f);
  %s
}
"""


@pytest.mark.parametrize("npairs", [2, 4, 8])
def test_equal_operands_have_registers_of_their_own(npairs, tmp_path):
    amp = [f"{c}{k}" for k in range(npairs) for c in "xy"]
    # x of every pair after the first is y of the pair before it
    init = [f"{a} = y{int(a[1:]) - 1}" if a[0] == "x" and a != "x0" else f"{a} = p[threadIdx.x + {64 * i}]"
            for i, a in enumerate(amp)]
    src = tmp_path / "k.hip"
    src.write_text(KERNEL % (jit._rotation(npairs), ", ".join(init), npairs, ", ".join(amp),
                             " ".join(f"p[threadIdx.x + {64 * i}] = {a};" for i, a in enumerate(amp))))
    out = tmp_path / "k.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "-S", "--offload-device-only", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    block = out.read_text().split("#ASMSTART")[1].split("s_branch 2f")[0]
    fma = re.findall(r"v_fma_f32 (v\d+), -(v\d+), (v\d+), (v\d+)", block)  # x', t, y, x of every component
    assert len(fma) == 2 * npairs
    regs = {fma[0][1]}
    assert all(t == fma[0][1] for _r, t, _y, _x in fma)
    for r, _t, y, x in fma:
        for v in (r, y, x):
            assert v not in regs, f"{v} holds two operands"
            regs.add(v)
