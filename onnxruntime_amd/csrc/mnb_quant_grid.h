// How the quantiser's workgroups are dealt out over a matrix of `strips` strips of 128 columns and `groups` groups of blocks
// along K, shared by host and device code.
//
// run = 0: strips side by side (grid.x), groups in grid.y.  Else each XCD takes a contiguous run of tiles, `run` groups of a
// strip one after the other, so that the pieces that they write side by side along K (scales, zero points, short blobs) meet
// in one level-2 cache and leave it as whole lines; all tiles are in grid.x then.
#pragma once
#include "mnb_layout.h"

struct MnbQuantTile {
  int64_t strip, group;
};

// The tile of workgroup x of `total` (run > 0).
MNB_HD MnbQuantTile mnb_quant_run_tile(unsigned x, unsigned total, int strips, int groups, int run) {
  const unsigned xcd = x & 7, odd = total & 7;
  const unsigned t = xcd * (total >> 3) + (xcd < odd ? xcd : odd) + (x >> 3);
  const unsigned band = t / ((unsigned)run * strips), first = band * run, rest = t - first * strips;
  const unsigned left = (unsigned)groups - first, height = (unsigned)run < left ? (unsigned)run : left;
  return {rest / height, first + rest % height};
}

struct MnbQuantGrid {
  unsigned x, y;
  int run;
  bool ok;  // a launch can hold it
};

// A launch holds 65536 workgroups in y, and fewer than 2^32 threads in x: runs, whose tiles are all in x, give way to
// strips side by side beyond that.
MNB_HD MnbQuantGrid mnb_quant_grid(int64_t strips, int64_t groups, int threads, bool runs) {
  const int64_t tiles = strips * groups;
  if (tiles >= ((int64_t)1 << 32) / threads) runs = false;
  MnbQuantGrid g{(unsigned)strips, (unsigned)groups, 0, groups <= 65536};
  if (runs) g.x = (unsigned)tiles, g.y = 1, g.run = 16;
  return g;
}
