// Layout of the copy in which lstm_resident_kernel's workgroups hand h to each other: [k / 4][columns][4] floats, the
// columns padded to eight.  Plain C++, so that it can be checked without a device.
//
// The kernel reads this copy with ordinary loads and never invalidates a cache, which is sound only if a 128-byte line
// belongs to one (row tile, column tile), that is to one producer and one flag: a reader that has seen the flag then brings
// in a line that is complete.  A row tile is 8 k = two k-blocks of columns * 16 bytes, a column tile starts at a multiple of
// 16 columns = 256 bytes inside a k-block: both are whole lines when the columns are a multiple of eight.  (A multiple of
// four is enough for one column tile; with more of them every other k-block then starts in the middle of a line, and that
// line holds columns of two tiles.)
#pragma once

constexpr int kResidentRows = 8;  // hidden rows per workgroup

constexpr int zr_resident_columns(int mb) { return (mb + 7) & ~7; }
// floats of one hidden state (one layer, one time step): an even number of row tiles, two of which are a k-group of the
// kernel's 16-column form
constexpr long long zr_resident_slot(int H, int mb) {
  return (long long)((H + 2 * kResidentRows - 1) / (2 * kResidentRows)) * (2 * kResidentRows) * zr_resident_columns(mb);
}
// element (row k, column n) of a state; `columns` as above
constexpr unsigned zr_resident_at(int k, int n, int columns) { return (unsigned)(((k >> 2) * columns + n) * 4 + (k & 3)); }

// An embedding column of H values is read in `blocks` k-blocks of four; those that reach past its end or lie behind it are
// moved down to end at H - 1 and read again what another block has read.  The part of weight k in block `block`, as the
// number of times it is halved: the readers of one k, the block it lies in first and then the moved ones, have 1/2, 1/4, ...
// of it and the last of them what is left.  The parts are powers of two and add up to one (to 2^-53, beyond 60 halvings).
constexpr int zr_resident_embed_halvings(int H, int blocks, int block, int k) {
  const int whole = H / 4;                 // blocks that lie inside the column as a whole
  const int here = k < 4 * whole ? 1 : 0;  // k is also read where it lies
  const int readers = k < H - 4 ? 1 : here + blocks - whole;
  const int mine = block < whole ? 0 : here + block - whole;
  const int halvings = mine < readers - 1 ? mine + 1 : readers - 1;
  return halvings < 60 ? halvings : 60;
}
