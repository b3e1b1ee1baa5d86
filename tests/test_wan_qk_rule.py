"""CPU test of the rule that gives a call to the one-pass q / k producer (csrc/wan_qk_rule.h,
compiled with the host compiler): never where it was measured slower than the two passes."""
import subprocess

import pytest

from icsa_hip import build

pytestmark = pytest.mark.cpu

MAIN = """
#include <cstdio>
#include "wan_qk_rule.h"
int main() {
  long long n; int H, sums;
  while (std::scanf("%lld %d %d", &n, &H, &sums) == 3) std::printf("%d\\n", (int)wan_one_pass(n, H, sums != 0));
}
"""

# (workgroups, heads, block sums): time of the two passes over the one pass's, in one run
MEASURED = {
    (4096, 3, 1): 0.68, (4096, 4, 1): 0.87, (2732, 5, 1): 0.98, (3900, 5, 1): 0.99,
    (586, 21, 1): 0.74, (1170, 21, 1): 0.91, (1366, 21, 1): 0.97, (1170, 22, 1): 0.94, (1170, 23, 1): 0.96,
    (624, 24, 1): 0.83, (664, 24, 1): 0.90, (702, 24, 1): 0.97, (624, 25, 1): 0.84, (684, 25, 1): 0.94,
    (546, 28, 1): 0.94, (634, 28, 1): 0.96, (518, 30, 1): 0.90, (528, 32, 1): 0.96, (312, 40, 1): 0.95,
    (2048, 8, 1): 1.23, (1756, 8, 1): 1.20, (1366, 10, 1): 1.25, (1034, 12, 1): 1.13, (1044, 13, 1): 1.08,
    (878, 16, 1): 1.19, (616, 20, 1): 1.17, (976, 24, 1): 1.17, (1366, 24, 1): 1.12, (878, 28, 1): 1.19,
    (878, 32, 1): 1.21, (450, 36, 1): 1.19, (390, 40, 1): 1.15, (586, 40, 1): 1.14, (878, 40, 1): 1.25,
    (683, 24, 0): 1.13, (780, 24, 0): 1.18, (390, 40, 0): 1.24, (439, 40, 0): 1.43,
}


def test_rule_follows_the_measurements(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", build.CSRC_DIR, str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")],
                   check=True)
    out = subprocess.run([str(tmp_path / "main")], input="\n".join("%d %d %d" % c for c in MEASURED),
                         capture_output=True, text=True, check=True).stdout.split()
    wrong = [(c, r, o) for (c, r), o in zip(MEASURED.items(), out) if (r > 1) != (o == "1")]
    assert not wrong, wrong
