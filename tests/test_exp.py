"""nc_expf_upto100 (csrc/nc_exp.h) gives nc_expf's bits: every 1021st float and every edge, on the host.

(All of them were compared when it was written: ten seconds on 8 cores with hardware fma.)
"""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "nanocompile_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <string.h>
#include <initializer_list>
#include "nc_exp.h"
static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static float value(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static long bad, seen;
static void check(uint32_t u) {
    const float x = value(u);
    if (x > 100.0f) return;
    const float want = nc_expf(x), got = nc_expf_upto100(x);
    ++seen;
    if (bits(want) != bits(got) && !(want != want && got != got)) ++bad;
}
int main() {
    for (uint64_t u = 0; u < 0x100000000ull; u += 1021) check((uint32_t)u);
    const float edges[] = {0.0f, -0.0f, 100.0f, -104.0f, -103.97f, -87.33655f, 88.72284f, 1.0f, -1.0f, 3e38f, -3e38f};
    for (float e : edges)
        for (int d = -2000; d <= 2000; ++d) check(bits(e) + (uint32_t)d);
    for (uint32_t top : {0x7f800000u, 0xff800000u, 0x7fc00000u, 0xffc00001u}) check(top);
    for (int k = -9700; k <= 9300; ++k)          // halfway between neighbours of the reduction's grid
        for (int d = -3; d <= 3; ++d) check(bits((float)((k + 0.5) * 0.010830424696249145)) + (uint32_t)d);
    printf("%ld %ld\n", seen, bad);
    return 0;
}
"""


def test_the_short_exp_is_nc_expf(tmp_path):
    source, binary = tmp_path / "exp.cpp", tmp_path / "exp"
    source.write_text(PROGRAM)
    cxx = shutil.which("g++") or "c++"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", f"-I{CSRC}", "-o", str(binary), str(source), "-lm"],
                   check=True)
    seen, bad = map(int, subprocess.run([str(binary)], check=True, capture_output=True, text=True).stdout.split())
    assert seen > 3_000_000 and bad == 0
