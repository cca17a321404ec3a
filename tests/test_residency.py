"""Workgroups that a cooperative launch counts on are there, however the
ordinary launches of other plans lie on the compute units (host arithmetic of
rb_residency.h, compiled here; no device)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "recblock-sptrsv_amd", "csrc")
LDS = 160 * 1024
STAGED = 99096                    # k_staged<1, double>
FUSED = [33560, 38000, 50000, 81000, LDS]  # k_fused by record format, and up

PROGRAM = """
#include <cstdio>
#include "rb_residency.h"
int main(int, char **v) {
    int a[3];
    while (std::scanf("%d %d %d", a, a + 1, a + 2) == 3)
        std::printf("%d %d %d\\n", rb::resident_slots(a[0], a[1], a[2]),
                    rb::small_grid(a[1]), rb::kSmallStreams);
}
"""


@pytest.fixture(scope="module")
def slots(tmp_path_factory):
    d = tmp_path_factory.mktemp("residency")
    (d / "m.cpp").write_text(PROGRAM)
    exe = str(d / "m")
    subprocess.run(["g++", "-std=c++17", "-I" + CSRC, str(d / "m.cpp"), "-o", exe], check=True)

    def call(per_cu, ncu, others):
        out = subprocess.run([exe], input="%d %d %d\n" % (per_cu, ncu, others),
                             capture_output=True, text=True, check=True).stdout
        return [int(t) for t in out.split()]
    return call


@pytest.mark.parametrize("ncu", [256, 64])
@pytest.mark.parametrize("mine", FUSED)
@pytest.mark.parametrize("theirs", [STAGED] + FUSED)
def test_slots_are_resident(slots, ncu, mine, theirs):
    per_cu = LDS // mine
    for others in range(slots(per_cu, ncu, 0)[2] + 1):
        promised, grid, _ = slots(per_cu, ncu, others)
        # every number of their workgroups on a compute unit that fits
        for each in range(1, LDS // theirs + 1):
            held = -(-others * grid // each)
            free = (ncu - held) * per_cu + held * ((LDS - each * theirs) // mine)
            assert promised <= free, (others, each)
