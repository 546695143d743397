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
// floats of one hidden state (one layer, one time step)
constexpr long long zr_resident_slot(int H, int mb) {
  return (long long)((H + kResidentRows - 1) / kResidentRows) * kResidentRows * zr_resident_columns(mb);
}
// element (row k, column n) of a state; `columns` as above
constexpr unsigned zr_resident_at(int k, int n, int columns) { return (unsigned)(((k >> 2) * columns + n) * 4 + (k & 3)); }
