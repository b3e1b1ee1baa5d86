"""CPU tests of how the flash kernel's items are dealt out (csrc/flash_plan.h, compiled with the
host compiler)."""
import heapq
import os
import subprocess

import pytest

from icsa_hip import build

pytestmark = pytest.mark.cpu

CUS = 256
START = 3                      # a workgroup's start, in tiles
COMBINE = 8                    # the sums of split items: 9-13 us, a tile 1.7 us

MAIN = """
#include <cstdio>
#include "flash_plan.h"
int main() {
  long long n; int tiles, split;
  while (std::scanf("%lld %d %d", &n, &tiles, &split) == 3) {
    const FlashPlan f = flash_plan(n, tiles, split != 0);
    std::printf("%d %d %d %d %lld %lld\\n", f.n_whole, f.bundle, f.n_bundle, f.n_chunk, (long long)f.part_bytes,
                (long long)flash_part_bytes_max(tiles));
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
    return dict(zip(GRID, ([int(x) for x in line.split()] for line in out.splitlines())))


def _span(lengths):
    """Makespan in tiles of workgroups of these lengths, each CU taking the next when it is free."""
    cu = [0.0] * CUS
    for x in lengths:
        heapq.heapreplace(cu, cu[0] + x + START)
    return max(cu)


def test_plan_covers_the_items(plans):
    for (n, tiles, split), (whole, bundle, n_bundle, chunks, part, part_max) in plans.items():
        assert bundle >= 1 and (n_bundle - 1) * bundle < max(whole, 1) <= max(n_bundle * bundle, 1)
        if chunks == 0:
            assert whole == n and part == 0
        else:                                   # a chunk holds tiles of at most two items
            assert split and n - whole <= chunks <= CUS
            assert 0 < part <= part_max


def test_plan_is_no_slower_than_an_item_a_workgroup(plans):
    """Several items a workgroup, or the last round's cut up, take no more time than one whole item
    a workgroup (2 %): 768 items of 256 tiles took 1,590 us in pairs, 1,390 us one by one."""
    slow = []
    for (n, tiles, split), (whole, bundle, n_bundle, chunks, part, part_max) in plans.items():
        lengths = [min(bundle, whole - i * bundle) * tiles for i in range(n_bundle)]
        lengths += [(n - whole) * tiles / max(chunks, 1)] * chunks
        t = _span(lengths) + (COMBINE if chunks else 0)
        if t > 1.02 * _span([tiles] * n):
            slow.append((n, tiles, split, bundle, round(t / _span([tiles] * n), 3)))
    assert not slow, slow
