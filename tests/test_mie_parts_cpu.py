"""Scratch of the homogeneous batch's three parts (gm_parts.h), compiled for the host:
the long series' part keeps the wavefronts that the budget holds, as a launch waits
for it; nothing exceeds the budget."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r"""
#include <stdio.h>
#include "gm_parts.h"
int main() {
  unsigned long long b, bs, ms, ss;
  long long w[3];
  while (scanf("%llu %lld %lld %lld %llu %llu %llu", &b, w, w + 1, w + 2, &bs, &ms, &ss) == 7) {
    const gm::HomogParts p = gm::homog_parts(b, {w[0], w[1], w[2], 0}, bs, ms, ss);
    printf("%lld %lld %lld %llu\n", (long long)p.big, (long long)p.mid, (long long)p.small,
           (unsigned long long)p.bytes);
  }
}
"""


@pytest.fixture(scope="module")
def parts(tmp_path_factory):
    d = tmp_path_factory.mktemp("parts")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "parts")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "geosmie_amd", "csrc"),
                    str(d / "main.cpp"), "-o", exe], check=True)

    def run(*args):
        out = subprocess.run([exe], input=" ".join(str(a) for a in args), capture_output=True,
                             text=True, check=True).stdout
        return [int(v) for v in out.split()]
    return run


SLOT = 64 * 3 * 8            # bytes of a row of 64 lanes
MID, SMALL = 14 * SLOT, 12 * SLOT


@pytest.mark.parametrize("rows, lanes, n, mid", [
    (2149, 64, 40000, True), (2149, 64, 200000, True), (8082, 64, 40000, True),
    (430, 32, 20000, False), (20100, 64, 200000, True), (60, 16, 3000, False),
    (1300000, 64, 10000, True)])
@pytest.mark.parametrize("budget", [3 << 30, 128 << 20, 125 << 20, 1 << 20, 30000])
def test_parts(parts, rows, lanes, n, mid, budget):
    lcap, resident = -(-rows // lanes), 2048
    slot = lcap * SLOT
    want = [min(-(-n * lanes // 64), resident), min(-(-n // 4), resident) if mid else 0,
            min(-(-n // 16), resident)]
    big, m, s, total = parts(budget, *want, slot, MID, SMALL)
    alone = max(1, min(want[0], budget // slot))    # what the budget holds without the others
    assert total == big * slot + m * MID + s * SMALL
    assert 1 <= big <= want[0] and 0 <= m <= want[1] and 0 <= s <= want[2]
    assert total <= max(budget, slot)
    # a sixteenth of the budget, or a block of each, is what the others may cost it
    assert big >= min(alone, (budget - max(budget // 16, MID + SMALL)) // slot)
    if want[0] * slot + want[1] * MID + want[2] * SMALL <= budget:
        assert [big, m, s] == want
    if budget >= slot + MID + SMALL:
        assert s >= 1 and (m >= 1) == mid
