"""Which walks take a label axis as blocks side by side: the rules of rnnt_blocks.h, compiled for the
host.  The shapes are ones that were measured both ways (one workgroup an utterance, blocks), on
either side of each line."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "rnnt_blocks.h"
using namespace rnnt;

int main(int argc, char** argv) {
  const Dims d = make_dims(atoi(argv[1]), atoi(argv[2]), atoi(argv[3]), 8, 0);
  int waves = 0;
  const int beta = beta_blocks(d, &waves);
  printf("%d %d %d %d", alpha_blocks(d), beta, beta > 1 ? waves : 0, viterbi_blocks(d));
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    where = tmp_path_factory.mktemp("blocks")
    source, out = str(where / "blocks.cpp"), str(where / "blocks")
    with open(source, "w") as f:
        f.write(PROGRAM)
    subprocess.check_call(["hipcc", "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                           "-I", os.path.join(ROOT, "transducer_amd", "csrc"), source, "-o", out])
    return out


def blocks(program, B, T, U):
    out = subprocess.run([program, str(B), str(T), str(U)], check=True, timeout=60,
                         stdout=subprocess.PIPE).stdout
    return tuple(int(x) for x in out.split())


# alpha's blocks, dalpha's with the wavefronts of one, the best path's
@pytest.mark.parametrize("B,T,U,want", [
    # short lattices of batches that fill the device with one workgroup an utterance: that way is
    # faster (alpha 131 against 168 us at B=256 T=100, 257 positions; dalpha 147 against 204 at B=162
    # T=200, 512; best path 143 against 170 at B=256 T=400, 300)
    (256, 100, 257, (1, 3, 2, 1)), (162, 100, 401, (1, 1, 0, 1)), (162, 200, 512, (1, 1, 0, 1)),
    (256, 400, 300, (1, 3, 2, 1)), (200, 999, 300, (1, 3, 2, 2)), (225, 100, 1000, (1, 1, 0, 1)),
    (162, 20, 1000, (4, 1, 0, 1)), (170, 300, 256, (1, 1, 0, 1)), (97, 300, 201, (1, 1, 0, 1)),
    # with a CU for every block, on long lattices, or where the other way is out of room
    (128, 100, 401, (2, 2, 4, 2)), (64, 100, 401, (2, 4, 2, 2)), (8, 10000, 401, (2, 4, 2, 2)),
    (200, 1000, 300, (2, 3, 2, 2)), (256, 100, 513, (3, 3, 4, 1)), (170, 300, 700, (3, 3, 4, 1)),
    (300, 100, 700, (3, 3, 4, 1)), (200, 300, 1000, (4, 1, 0, 1)), (48, 300, 1000, (4, 8, 2, 4)),
    (128, 300, 201, (1, 2, 2, 1)), (32, 2000, 201, (1, 2, 2, 1)), (8, 2000, 201, (1, 1, 0, 1)),
    (200, 12500, 401, (2, 2, 4, 2)), (256, 500, 640, (3, 3, 4, 1)), (225, 1000, 1000, (4, 1, 0, 1)),
    # axes past 1024 positions, whatever the batch, and past 16 blocks
    (300, 50, 1100, (5, 5, 4, 5)), (8, 50, 1100, (5, 9, 2, 5)), (8, 50, 4000, (16, 16, 4, 16)),
    (8, 50, 4097, (1, 1, 0, 1)), (8, 50, 100, (1, 1, 0, 1)),
])
def test_blocks_side_by_side(program, B, T, U, want):
    assert blocks(program, B, T, U) == want
