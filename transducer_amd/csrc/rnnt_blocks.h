// How the lattice walks deal a label axis to workgroups: host code without the device's, so that
// the rules can be read, and tested, by themselves.
//
// Up to 256 positions one workgroup takes them, one a lane.  Up to 1024 there are two ways: blocks
// of the axis side by side, a workgroup each with one position a lane (alpha_walk_kernel and its
// like), or one workgroup with two or four positions a lane (alpha_kernel and its like).  Blocks
// take a step in a third to two thirds of the time, so they win as long as every workgroup
// has a CU to itself; past that they share issue slots among themselves, and what the hand-over adds
// and the delay from block to block (as many steps as a block has positions) are a loss on short
// lattices.  Measured with utterances at full length, both ways from the same tree: 30 to 4000
// frames, 65 to 512 utterances, 257 to 1000 positions; the figures below are time of one workgroup
// over time of blocks.  (Ragged batches favour blocks more: utterances leave blocks empty.)
#pragma once

#include <algorithm>

#include "rnnt_internal.h"

namespace rnnt {

// Label positions one launch of a several-positions-a-lane walk covers: the whole axis up to 1024, else
// blocks of 1024 (64 lanes x 16 positions), one launch per block.
inline int block_cells_per_lane(const Dims& d) { return std::min(cells_per_lane(d.U), 16); }
inline int label_blocks(const Dims& d) {
  const int width = 64 * block_cells_per_lane(d);
  return (d.U + width - 1) / width;
}

// Blocks of 256 label positions that the alpha walk runs side by side (1: none).
//   two      256 workgroups (1.30 .. 2.10); up to 512 from 1000 frames on (1.04 .. 1.16, below that
//            0.77 .. 1.35, on 257 positions 0.77 .. 0.99)
//   three    900 workgroups (0.99 .. 3.42)
//   four     800 workgroups (1.11 .. 3.16); up to 900 from 1000 frames on (1.04, below 0.88 .. 1.31)
// Past 1024 positions the other way is a launch per 1024, many times slower whatever the batch;
// workgroups beyond the device's CUs queue in order.
inline int alpha_blocks(const Dims& d) {
  const int n = (d.U + 255) / 256;
  if (n < 2 || n > 16) return 1;
  if (d.U > 1024) return n;
  const long workgroups = (long)d.B * n;
  const int alone = n == 2 ? 256 : n == 3 ? 900 : 800, at_length = n == 2 ? 512 : 900;
  return workgroups <= (d.T >= 1000 ? at_length : alone) ? n : 1;
}

// Blocks that the dalpha walk runs side by side, and the wavefronts (64 positions each) of a block.
// A cell is six instructions and 12 bytes, and what one CU's memory path moves holds the walk, so
// blocks of 128 positions are the better ones where there is a CU for each (B=8 T=10000, 401
// positions: 610 us with blocks of 256, 372 with 128).
//   129 .. 256   (four wavefronts of one workgroup can take them as well) two of 128 up to 256
//                workgroups, where the walk's planes are more than the memory-side cache keeps
//                beside everything else: 80 MB of cells, 130 on short lattices (1.01 .. 1.61; below,
//                and with more workgroups, 0.51 .. 1.10)
//   .. 384       three of 128 for any batch (0.94 .. 2.60, one of 120 figures below 1)
//   .. 512       four of 128 up to 256 workgroups, then two of 256 up to 256 (1.11 .. 1.59; with more
//                0.80 .. 1.24, of 128 0.78 .. 1.26)
//   .. 768       of 128 up to 512 workgroups, then three of 256 up to 900 (1.10 .. 2.54)
//   .. 1024      of 128 up to 512 workgroups, then four of 256 up to 400 (0.96 .. 1.52; with more
//                0.74 .. 1.54)
// One workgroup of 385 .. 512 positions takes four wavefronts, whose three hand-over arrays have to fit
// LDS; longer utterances go as blocks.
inline int beta_blocks(const Dims& d, int* waves) {
  const int n2 = (d.U + 127) / 128, n4 = (d.U + 255) / 256;
  const long B = d.B;
  *waves = 2;
  if (d.U <= 128) return 1;
  if (d.U <= 256) {
    const unsigned long long planes = 12ull * d.B * d.U * d.Dp;
    return B <= 128 && planes > (d.Dp < 700 ? 130ull : 80ull) * 1000000 ? 2 : 1;
  }
  if (n2 <= 16 && (d.U <= 384 || B * n2 <= (d.U <= 512 ? 256 : 512))) return n2;
  *waves = 4;
  if (d.U <= 512) return B <= 128 || d.Dp > 12288 ? 2 : 1;
  if (d.U <= 768) return B * 3 <= 900 ? 3 : 1;
  if (d.U <= 1024) return B * 4 <= 400 ? 4 : 1;
  return n4 <= 16 ? n4 : 1;
}

// ---- best path
// 32-step words per column of the decision table (one spare)
inline int viterbi_words(const Dims& d) { return (d.T + d.U + 31) / 32 + 1; }
// One workgroup with several positions a lane: its wavefronts (four, or two, if their hand-over
// arrays fit LDS beside an int per label position) and LDS, with the decision columns in it if they fit
// too (one launch only: with several, every block's columns must be there for the backtrace of
// the last).
struct ViterbiOne {
  int wavefronts;
  bool columns;
  size_t lds;
};
inline ViterbiOne viterbi_one(const Dims& d) {
  const int cpl = block_cells_per_lane(d);
  const bool single = label_blocks(d) == 1;
  const size_t taken = sizeof(int) * (size_t)((d.U + 3) & ~3), hand = sizeof(float) * (size_t)d.Dp;
  ViterbiOne r;
  r.wavefronts = single && cpl >= 4 && taken + 3 * hand <= 144 * 1024 ? 4
                 : cpl >= 2 && taken + hand <= 144 * 1024 ? 2 : 1;
  r.lds = taken + (r.wavefronts - 1) * hand;
  const size_t columns = sizeof(unsigned) * (size_t)64 * cpl * viterbi_words(d);
  r.columns = single && r.lds + columns <= 60 * 1024;
  if (r.columns) r.lds += columns;
  return r;
}
// Blocks of 256 label positions that the best-path walk runs side by side (1: none).
//   two      256 workgroups (1.06 .. 2.00); up to 512 where one workgroup has no room for the decision
//            columns in LDS and traces the path from memory (1.08 .. 1.51; with room 0.83 .. 0.95)
//   more     192 workgroups, which keeps the decode's scratch at what it is for larger batches.
//            (Not for speed: 1.24 .. 2.47 for every batch.)
inline int viterbi_blocks(const Dims& d) {
  const int n = (d.U + 255) / 256;
  if (n < 2 || n > 16) return 1;
  if (d.U > 1024) return n;
  const long workgroups = (long)d.B * n;
  if (n == 2) return workgroups <= 256 || (workgroups <= 512 && !viterbi_one(d).columns) ? 2 : 1;
  return workgroups <= 192 ? n : 1;
}

}  // namespace rnnt
