"""The registers of the walk's plain steps. The block of steps writes its
read-write operands while it still reads its inputs, so no input may share a
register with one of them, also where the caller passes the same value for
both (a shared register is the compiler's right unless the operands are marked
early-clobber). Compiled for the device, read in the listing of this code."""
import re
import subprocess

import pytest

from newrecon_amd.build import CSRC, HIPCC, HIPFLAGS

SOURCE = """
#include "walk_steps.h"
extern "C" __global__ void steps(const float* f, const uint32_t* u, float* out) {
    const int i = threadIdx.x;
    float xn = f[i], yn = f[i + 64], zn = f[i + 128], at = f[i + 192], cur = f[i + 256];
    uint32_t px = u[i], py = u[i + 64], pz = u[i + 128];
    float seg[4];
    uint32_t off[4];
    ostr::plain_steps(xn, yn, zn, px, py, pz, at, cur, %s, seg, off);
    float s = xn + yn + zn + at + cur;
    uint32_t t = px + py + pz;
    for (int k = 0; k < 4; ++k) s += seg[k], t += off[k];
    out[i] = s + (float)t;
}
"""
# xi, yi, zi, xs, ys, zs, len
INPUTS = {
    "own": "f[i + 320], f[i + 384], f[i + 448], u[i + 192], u[i + 256], u[i + 320], f[i + 512]",
    "next-crossings": "xn, yn, zn, px, py, pz, f[i + 512]",
    "positions": "at, cur, at, px, px, px, cur",
}


@pytest.mark.parametrize("inputs", INPUTS)
def test_inputs_keep_their_registers(tmp_path, inputs):
    src, asm = tmp_path / "steps.hip", tmp_path / "steps.s"
    src.write_text(SOURCE % INPUTS[inputs])
    subprocess.run([HIPCC, *HIPFLAGS, "-I", CSRC, "--offload-device-only", "-S", str(src), "-o",
                    str(asm)], check=True, capture_output=True)
    block = asm.read_text().split("#ASMSTART")[1].split("#ASMEND")[0]
    written, read = set(), set()
    for line in block.splitlines():
        m = re.match(r"\s*v_(\w+) (.*)", line)
        if not m:
            continue
        regs = re.findall(r"\bv\d+\b", m.group(2))
        if m.group(1).startswith("cmpx"):
            read.update(regs)
        else:
            written.add(regs[0])
            read.update(regs[1:])
    # 8 read-write operands, 4 segments, 4 offsets; 7 inputs, which nothing writes
    assert len(written) == 16
    distinct = len(set(re.findall(r"[^,]+", INPUTS[inputs].replace(" ", ""))))
    assert len(read - written) == distinct
