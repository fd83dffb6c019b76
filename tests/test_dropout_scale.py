"""The factor that replaces dropout's division for 16-bit values (CPU: dropout_scale of thn_dropout.h in a host program).  Where there is
one, its product rounds like the quotient for every value of the type, and most probabilities have one."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "triton-hub_amd", "csrc")
PROGRAM = r"""
#include <stdio.h>
#include "thn_dropout.h"
using namespace thn;
static float wide(uint32_t bits, int dtype) {
    float v;
    if (dtype == kBF16) { bits <<= 16; memcpy(&v, &bits, 4); return v; }
    const uint16_t half = static_cast<uint16_t>(bits);
    _Float16 h;
    memcpy(&h, &half, 2);
    return static_cast<float>(h);
}
static uint32_t narrow(float v, int dtype) {
    if (dtype == kBF16) { uint32_t u; memcpy(&u, &v, 4); return (u + 0x7fffu + (u >> 16 & 1u)) >> 16; }
    const _Float16 h = static_cast<_Float16>(v);
    uint16_t u;
    memcpy(&u, &h, 2);
    return u;
}
static int found = 0, wrong = 0;
static void check(float p, int dtype) {
    const float keep = 1.0f - p, scale = dropout_scale(keep, dtype);
    if (scale == 0.0f) return;
    ++found;
    for (uint32_t bits = 0; bits < 65536u; ++bits) {
        const float x = wide(bits, dtype);
        if (x == x && narrow(x / keep, dtype) != narrow(x * scale, dtype)) { ++wrong; printf("p = %.9g value %u\n", p, bits); return; }
    }
}
int main() {
    for (const int dtype : {kF16, kBF16}) {
        found = wrong = 0;
        for (int i = 1; i < 100; ++i) check(static_cast<float>(i) / 100.0f, dtype);
        printf("%d %d %d\n", dtype == kF16 ? 16 : 17, found, wrong);
        for (int i = 0; i < 200; ++i) check(static_cast<float>(i * 4 + 1) / 1009.0f, dtype);
        for (int e = 1; e <= 24; ++e) { check(ldexpf(1.0f, -e), dtype); check(1.0f - ldexpf(1.0f, -e), dtype); check(1.0f - ldexpf(1.3f, -e), dtype); }
        printf("%d %d %d\n", dtype == kF16 ? 26 : 27, found, wrong);
        if (dropout_scale(0.0f, dtype) != 0.0f || dropout_scale(1.0f, dtype) != 1.0f || dropout_scale(0.5f, dtype) != 2.0f) ++wrong;
    }
    if (dropout_scale(0.5f, kF32) != 0.0f || dropout_scale(0.5f, kF64) != 0.0f) ++wrong;
    return wrong;
}
"""


def test_products_round_like_quotients(tmp_path):
    source, program = tmp_path / "scale.hip", tmp_path / "scale"
    source.write_text(PROGRAM)
    subprocess.check_call(["hipcc", "--offload-host-only", "-O2", "-std=c++17", "-w", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                           str(source), "-o", str(program)])
    done = subprocess.run([str(program)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout
    counts = {int(kind): (int(found), int(wrong)) for kind, found, wrong in (line.split() for line in done.stdout.splitlines())}
    assert counts[16] == (86, 0) and counts[17] == (92, 0)         # of p = 0.01, 0.02 .. 0.99
    assert counts[26][1] == 0 and counts[27][1] == 0
