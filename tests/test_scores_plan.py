"""How the last-query scores' launches are cut (csrc/sp_scores_plan.h, plain host arithmetic): by the rows of the grid, which a group with
an odd number of heads has more of than its heads need, and never into more chunks than the workspace holds."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "shareprefill_amd", "csrc")
HEADS = [(1, 1), (7, 1), (14, 2), (16, 4), (28, 4), (32, 8), (32, 32), (9, 9), (10, 2), (40, 8), (64, 8), (128, 128), (6000, 6000)]
TOKENS = [128, 1500, 3001, 4500, 6177, 10007, 16384, 20000, 49000, 65001, 131072, 524288]
PROGRAM = """
#include <stdio.h>
#include "sp_scores_plan.h"
int main() {
  int hq, hkv;
  long n;
  while (scanf("%d %d %ld", &hq, &hkv, &n) == 3) {
    const long tiles = lq_ceil_div(n, 128), rows = lq_wg_rows(hq, hkv), t = lq_tiles_per_wg(tiles, rows);
    printf("%ld %ld %ld %ld\\n", rows, t, lq_ceil_div(tiles, t), (long)lq_max_chunks(tiles, hq));
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """{(hq, hkv, n): (rows, tiles per workgroup, chunks, chunks the workspace holds)}"""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    tmp = tmp_path_factory.mktemp("plan")
    (tmp / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-Wall", "-Werror", "-Wno-unused-function", "-I", CSRC, str(tmp / "plan.cpp"), "-o", str(tmp / "plan")], check=True)
    keys = [(hq, hkv, n) for hq, hkv in HEADS for n in TOKENS]
    out = subprocess.run([str(tmp / "plan")], input="".join("%d %d %d\n" % k for k in keys), capture_output=True, text=True, check=True).stdout
    return dict(zip(keys, (tuple(map(int, l.split())) for l in out.splitlines())))


def test_launches_of_as_many_workgroups_are_cut_alike(plans):
    for n in TOKENS:
        assert plans[28, 4, n][:3] == plans[32, 8, n][:3]  # 16 rows either way: seven heads take four workgroups
        assert plans[14, 2, n][:3] == plans[16, 4, n][:3]
        assert plans[32, 32, n][:3] == plans[64, 8, n][:3]  # a head each: half the workgroup stands empty
    # at 49000 tokens 28 / 4 heads, cut for 14 rows, ran 560 workgroups of 11 tiles, a second round of 48 (184 us; 166 before, 512 now)
    assert plans[28, 4, 49000][:3] == (16, 12, 32)


def test_the_workspace_holds_every_cut(plans):
    for key, (_, tiles, chunks, room) in plans.items():
        assert 1 <= tiles <= 32 and chunks <= room, key
