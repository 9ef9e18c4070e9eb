"""The branch generator switches the rounding mode around its fma
(ctc_amd/csrc/udx_dev.h); two writes of the mode register need two
instructions (or wait states) between them.  Checked on the code the compiler
makes of chains that follow one another, in a small kernel each and with the
library's flags."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ctc_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = """
#include "udx_dev.h"
using namespace udx;
extern "C" __global__ void pairs(float *x) {
    float *p = x + 4 * threadIdx.x;
    float a = p[0], b = p[1], c = p[2], d = p[3];
    logistic18x2(&a, &b);
    logistic18x2(&c, &d);
    p[0] = a; p[1] = b; p[2] = c; p[3] = d;
}
extern "C" __global__ void mixed(float *x) {
    float *p = x + 5 * threadIdx.x;
    float a = p[0], b = p[1], c = p[2], d = p[3], e = p[4];
    logistic18x2(&a, &b);
    c = logistic18(c);
    logistic18x2(&d, &e);
    p[0] = a; p[1] = b; p[2] = c; p[3] = d; p[4] = e;
}
extern "C" __global__ void singles(float *x) {
    float *p = x + 3 * threadIdx.x;
    const float a = p[0], b = p[1], c = p[2];
    p[0] = logistic18(a);
    p[1] = logistic18(b);
    p[2] = logistic18(c);
}
"""


def gaps(asm):
    """per kernel, the wait states between successive mode writes"""
    out, name, since = {}, None, None
    for line in asm.splitlines():
        line = line.strip()
        m = re.match(r"(\w+):", line)
        if m and not line.startswith((".", "L")):
            name, since = m[1], None
        if not line or line.startswith((";", ".")) or ":" in line.split()[0]:
            continue
        op = line.split()[0]
        if op.startswith("s_setreg") and "HW_REG_MODE" in line:
            if since is not None:
                out.setdefault(name, []).append(since)
            since = 0
        elif since is not None:
            since += int(line.split()[1], 0) + 1 if op == "s_nop" else 1
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_mode_writes_two_wait_states_apart(tmp_path):
    src, asm = tmp_path / "chains.hip", tmp_path / "chains.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-S", "--cuda-device-only", str(src),
                    "-o", str(asm)], check=True, stderr=subprocess.DEVNULL)
    g = gaps(asm.read_text())
    assert {k: len(v) for k, v in g.items()} == {"pairs": 35, "mixed": 53, "singles": 53}
    assert min(min(v) for v in g.values()) >= 2, g
