"""How many frames a plan's slots hold (csrc/group.h), compiled for the host: the group of a grid, the
caller's frame count, what stays free of the device's memory however many plans there are, and the
retries when an allocation fails."""
import os
import subprocess

import pytest

from conftest import PKG

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "group.h"
using namespace mdsf;
const size_t GB = (size_t)1 << 30, MB = (size_t)1 << 20;
int main(int argc, char** argv) {
  const int what = atoi(argv[1]);
  if (what == 0) {   // group_frames tiles frames bytes(MB) free(MB) total(MB) taken(MB)
    GroupMemory mem;
    mem.free = atoll(argv[5]) * MB;
    mem.total = atoll(argv[6]) * MB;
    mem.taken = atoll(argv[7]) * MB;
    printf("%d\n", group_frames(atoll(argv[2]), atoll(argv[3]), atoll(argv[4]) * MB, mem));
  } else if (what == 1) {   // plans of one size until one frame each does not fit
    const size_t bytes = atoll(argv[2]) * MB;
    GroupMemory mem;
    mem.free = mem.total = 288 * GB;
    int plans = 0;
    for (;; ++plans) {
      int g = group_frames(64, 0, bytes, mem);
      const int e = take_group(&g, 2, [&](int n) { return n * bytes <= mem.free ? 0 : 2; });
      if (e) break;
      mem.free -= g * bytes;
      mem.taken += (g - 1) * bytes;
    }
    printf("%d %d\n", plans, (int)(mem.total / bytes));
  } else {   // take_group: which groups are tried when `fit` frames fit
    int g = atoi(argv[2]);
    const int fit = atoi(argv[3]), other = atoi(argv[4]);
    const int e = take_group(&g, 2, [&](int frames) {
      printf("%d ", frames);
      return other ? 7 : (frames <= fit ? 0 : 2);
    });
    printf("| %d %d\n", g, e);
  }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("group")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(PKG, "csrc"),
                    str(d / "main.cpp"), "-o", exe], check=True)
    return lambda *a: subprocess.run([exe, *map(str, a)], check=True, capture_output=True,
                                     text=True).stdout.strip()


@pytest.mark.parametrize("tiles,frames,mb,free,total,taken,want", [
    (64, 0, 10, 0, 0, 0, 16),               # a 64^3 grid, memory unknown
    (64, 0, 10, 290000, 294912, 0, 16),
    (512, 0, 10, 290000, 294912, 0, 4),     # 128^3
    (2048, 0, 10, 290000, 294912, 0, 1),
    (4096, 0, 10, 290000, 294912, 0, 1),    # 256^3 fills the chip
    (1, 0, 10, 290000, 294912, 0, 16),
    (64, 1, 10, 290000, 294912, 0, 1),      # the caller's frames
    (64, 5, 10, 290000, 294912, 0, 5),
    (64, 100, 10, 290000, 294912, 0, 16),
    (64, 0, 300, 290000, 294912, 0, 6),     # 2 GiB of state
    (64, 0, 3000, 290000, 294912, 0, 1),
    (64, 0, 100, 140000, 294912, 0, 16),    # half of the memory in other use
    (64, 0, 100, 100 + 16 * 99, 294912, 0, 1),      # a sixteenth of what is free
    (64, 0, 100, 100 + 16 * 100, 294912, 0, 2),
    (64, 0, 100, 100 + 16 * 450, 294912, 0, 5),
    (64, 0, 100, 50, 294912, 0, 1),
    (64, 0, 100, 200000, 294912, 73728 - 250, 3),   # a quarter of the device for all groups
    (64, 0, 100, 200000, 294912, 73728, 1),
    (64, 0, 100, 200000, 294912, 90000, 1),
])
def test_group(rule, tiles, frames, mb, free, total, taken, want):
    assert int(rule(0, tiles, frames, mb, free, total, taken)) == want


@pytest.mark.parametrize("mb", [24, 140, 500, 2100])
def test_many_plans(rule, mb):
    """Plans whose one-frame states fill three quarters of the device fit, as without groups."""
    plans, whole = map(int, rule(1, mb).split())
    assert plans >= whole * 3 // 4


@pytest.mark.parametrize("group,fit,want", [(16, 16, "16 | 16 0"), (16, 5, "16 8 4 | 4 0"),
                                            (5, 1, "5 2 1 | 1 0"), (16, 0, "16 8 4 2 1 | 1 2"),
                                            (1, 0, "1 | 1 2")])
def test_retries(rule, group, fit, want):
    assert rule(2, group, fit, 0) == want


def test_other_errors_end_the_retries(rule):
    assert rule(2, 16, 16, 1) == "16 | 16 7"
