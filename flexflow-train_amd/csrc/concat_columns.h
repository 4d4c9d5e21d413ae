// How many columns of a concatenated row one workgroup of concat.hip takes (host code, no GPU headers).
#pragma once
#include <stdint.h>

namespace ffk {

constexpr int kConcatThreads = 256;

// A workgroup takes as many rows, of those there are, as it has threads for.  It takes all columns it can, or, where
// that leaves more than a 32nd fewer threads over, an even share of one more piece of the row and up to three more, or
// a power of two down to eight (288 columns of 16 bytes, nine parts of 128 floats: 9 x 32, where 256 + 32 had every
// other workgroup work with 32 threads; [16384, 9 x 128] 39 us, with four rows of a thread in flight 28, a copy of that
// size 25).  These widths take 0.04 us of a call's host time, where all 256 took 2.3 and left 2% fewer threads over.
inline int concat_columns(int64_t units_per_row, int64_t rows) {
  int64_t const fewest = (units_per_row + kConcatThreads - 1) / kConcatThreads;
  int64_t pieces = 0;  // of a row
  int cols = 0, each = 0;  // of a piece; rows of a workgroup
  auto offer = [&](int c, int64_t p, int e) {
    if (rows < e) e = (int)rows;
    // threads with an element, of those launched: units_per_row * e / (256 * p)
    if (cols == 0 || 32 * e * pieces > 33 * each * p) cols = c, each = e, pieces = p;
  };
  if (fewest > 8) return kConcatThreads;  // an uneven piece at the end is then a ninth at most
  int const units = (int)units_per_row, widest = units < kConcatThreads ? units : kConcatThreads;
  offer(widest, fewest, kConcatThreads / widest);
  for (int p = (int)fewest + 1; p <= (int)fewest + 4 && p <= units; p++) {
    int const c = (units + p - 1) / p;
    offer(c, (units + c - 1) / c, kConcatThreads / c);
  }
  for (int shift = 7; shift >= 3; shift--) offer(1 << shift, (units + (1 << shift) - 1) >> shift, kConcatThreads >> shift);
  return cols;
}

}  // namespace ffk
