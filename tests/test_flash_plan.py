"""CPU tests of how the flash kernel's items are dealt out (csrc/flash_plan.h, compiled with the
host compiler)."""
import heapq
import os
import subprocess

import pytest

from icsa_hip import build

pytestmark = pytest.mark.cpu

CUS, XCDS = 256, 8
START = 3                      # a workgroup's start, in tiles
COMBINE = 8                    # the sums of split items: 9-13 us, a tile 1.7 us

MAIN = """
#include <cstdio>
#include "flash_plan.h"
int main() {
  long long n; int tiles, split;
  while (std::scanf("%lld %d %d", &n, &tiles, &split) == 3) {
    const FlashPlan f = flash_plan(n, tiles, split != 0);
    std::printf("%d %d %lld %lld", f.n_whole, f.n_chunk, (long long)f.part_bytes,
                (long long)flash_part_bytes_max(tiles));
    for (int wg = 0; wg < FA_XCDS * f.n_bundle; ++wg) {
      const FlashRun r = flash_whole_run(wg, f.n_whole, f.n_bundle);
      std::printf(" %d %d", r.first, r.count);
    }
    std::printf("\\n");
  }
}
"""

GRID = [(n, t, s) for t in (1, 2, 8, 9, 12, 13, 18, 32, 64, 96, 128, 147, 160, 171, 200, 256, 300, 576)
        for n in (1, 2, 40, 100, 255, 256, 257, 300, 512, 640, 768, 1024, 1280, 1774, 1792, 2551, 3328, 5376, 10240)
        for s in (0, 1)]


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", build.CSRC_DIR, str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)
    out = subprocess.run([str(d / "main")], input="\n".join("%d %d %d" % g for g in GRID), capture_output=True,
                         text=True, check=True).stdout
    res = {}
    for g, line in zip(GRID, out.splitlines()):
        x = [int(y) for y in line.split()]
        res[g] = x[:4] + [list(zip(x[4::2], x[5::2]))]
    return res


def _span(lengths):
    """Makespan in tiles of workgroups of these lengths, each CU taking the next when it is free."""
    cu = [0.0] * CUS
    for x in lengths:
        heapq.heapreplace(cu, cu[0] + x + START)
    return max(cu)


def test_plan_covers_the_items(plans):
    for (n, tiles, split), (whole, chunks, part, part_max, runs) in plans.items():
        step = len(runs) // XCDS
        assert sorted(first + i * step for first, count in runs for i in range(count)) == list(range(whole))
        if chunks == 0:
            assert whole == n and part == 0
        else:                                   # a chunk holds tiles of at most two items
            assert split and n - whole <= chunks <= CUS
            assert 0 < part <= part_max


def test_neighbouring_items_run_side_by_side(plans):
    """The i-th items of an XCD's workgroups are consecutive: the items of a head share its K and
    V in that XCD's L2 (640 items of 64 tiles, two a head, one after the other in a workgroup:
    499 us a call, side by side 438)."""
    for whole, chunks, part, part_max, runs in plans.values():
        step = len(runs) // XCDS
        for x in range(XCDS):
            for i in range(max([c for _, c in runs[x::XCDS]], default=0)):
                at = [first + i * step for first, count in runs[x::XCDS] if count > i]
                assert at == list(range(at[0], at[0] + len(at)))


def test_plan_is_no_slower_than_an_item_a_workgroup(plans):
    """Several items a workgroup, or the last round's cut up, take no more time than one whole item
    a workgroup (2 %): 768 items of 256 tiles took 1,541 us in pairs, 1,350 one by one."""
    slow = []
    for (n, tiles, split), (whole, chunks, part, part_max, runs) in plans.items():
        t = _span([c * tiles for _, c in runs if c] + [(n - whole) * tiles / max(chunks, 1)] * chunks)
        t += COMBINE if chunks else 0
        if t > 1.02 * _span([tiles] * n):
            slow.append((n, tiles, split, round(t / _span([tiles] * n), 3)))
    assert not slow, slow
