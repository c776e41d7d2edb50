"""The lattice walks address an utterance's planes through buffers whose size is a 32-bit word and
which they move on every GiB.  Planes of 4 GiB and more are checked here by their numbers, in a
program of its own that takes them from the walks' own header; no device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "rnnt_internal.h"
using namespace rnnt;

int main(int argc, char** argv) {
  const Dims d = make_dims(1, atoi(argv[1]), atoi(argv[2]), 8, 0);
  const size_t group = 16 * (size_t)d.Ua, groups = d.Dp / 4, plane = group * groups;
  const size_t span = (1u << 30) / group;
  printf("plane of %zu bytes\n", plane);
  for (size_t origin = 0; origin < groups; origin += span) {
    const size_t left = plane - origin * group;
    const size_t size = buffer_bytes(left);
    if (size > left) return printf("%zu bytes of %zu from group %zu\n", size, left, origin), 1;
    // a window's own groups, and as many as a walk looks ahead of its last one
    for (size_t g = origin; g < groups && g < origin + span + 32; ++g)
      if ((g - origin + 1) * group > size)
        return printf("group %zu is outside the %zu bytes from group %zu\n", g, size, origin), 1;
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def windows(tmp_path_factory):
    where = tmp_path_factory.mktemp("windows")
    source, out = str(where / "windows.cpp"), str(where / "windows")
    with open(source, "w") as f:
        f.write(PROGRAM)
    subprocess.check_call(["hipcc", "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                           "-I", os.path.join(ROOT, "transducer_amd", "csrc"), source, "-o", out])
    return out


@pytest.mark.parametrize("T,U", [(260036, 2100), (258040, 4096), (523180, 1100), (2096844, 300),  # 2^32 bytes
                                 (16777206, 2), (16777300, 2), (8388500, 100), (8388700, 100),
                                 (6000000, 257), (100000000, 20), (2000, 100), (1, 1)])
def test_a_walks_buffer_holds_every_group_that_it_is_asked_for(windows, T, U):
    subprocess.run([windows, str(T), str(U)], check=True, timeout=60)
