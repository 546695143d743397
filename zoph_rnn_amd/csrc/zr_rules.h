// Which kernel a call takes, as plain C++ (no device code), so that a rule can be checked without a device against what was
// measured on both sides of its line (tests/test_rules_cpu.py holds the measurements).
#pragma once

// ---- one LSTM node: tiles of 4 or 8 hidden rows (zr_lstm_rows.hip) or launch_fused (zr_lstm.hip)

// launch_fused's time for a single fp32 node, us.  vec: H % 4 == 0 and 16-byte aligned inputs.  Follows its own choice of
// kernel; the constants are fitted to H = 300 .. 1500 at 64 .. 512 columns, two and three segments, and hold to about 10 %.
inline double zr_fused_node_us(int H, int mb, int nseg, bool vec, int cus) {
  const int j = (H + 31) / 32, n32 = (mb + 31) / 32;
  const int whole = j * ((n32 + 1) / 2);
  if (H % 8 == 0 && vec && whole < 200) {
    const int tiles = j * n32;
    int parts = (cus + tiles / 2) / tiles;
    if (parts > H / 128) parts = H / 128;
    if (parts > 8) parts = 8;
    if (parts >= 2) {  // K split across workgroups; the row tiles are dealt to the eight dies
      const int rounds = ((j + 7) / 8 * n32 * parts + cus / 8 - 1) / (cus / 8);
      return rounds * (6.5 + 0.8 * parts + 0.018 * H / parts * nseg);
    }
  } else if (vec && n32 >= 3 && whole < 200) {  // weights through LDS
    const int tiles = j * ((n32 + 3) / 4);
    int parts = cus / (tiles * nseg);
    if (parts > 8) parts = 8;
    if (parts < 1) parts = 1;
    const int rounds = (tiles * nseg * parts + cus - 1) / cus;
    return rounds * (12.5 + 0.075 * H / parts + 3.0 * parts);
  }
  const int tn = n32 >= 2 && whole > 128 ? 2 : 1;
  const int wgs = j * ((n32 + tn - 1) / tn);
  if (wgs < 192) return 0.033 * H * nseg * tn;
  return (wgs + cus - 1) / cus * (5.0 + (tn == 2 ? 0.036 : 0.0205) * H * nseg);
}

// Tile by size, one node of H = 1000 / 500 / 300 at up to 128 columns, us (the register-streaming kernel of zr_lstm.hip
// with K split across workgroups: 16-27 / 30-33 / 23-30):
//   4 x 16:  13.0 at 12 columns /  6.4 at 12, 8.6 at 37 /  5.5 at 20      8 x 16:  11.5 at 12, 12.0 at 32 / 7.4 at 37 / 6.1
//   8 x 32:  17.0 at 64 / 11.7 at 128 / 7.7 at 100                        8 x 64:  26.5 at 128 / 16.8 at 128
// The smallest tile that keeps the workgroups within one per compute unit wins, except that 4 x 16 tiles of H > 512 read the
// activations once too often (13.0 against 11.5).  Wide tiles of a long K range lose to the streaming kernel where that has
// its whole-group form (H = 2000, 64 columns: 71 against 48), and so does any second round of workgroups there (H = 1000, 192
// columns: 42-65 against 37).  For 8 x 64 tiles it is a matter of how well the older kernels' own tiles fit the chip: H =
// 1000, 128 columns 27.2 against 26.1 and 96 columns 25.9 against 36.3; H % 8 != 0, in rounds, H = 1001, 192 columns
// 54.5 against 43.5, H = 1100 56.8 against 94.2.
// Returns 0 = 4 rows x 16 columns, 1 = 8 x 16, 2 = 8 x 32, 3 = 8 x 64; -1: leave the node to launch_fused.
inline int zr_lstm_rows_shape(int H, int mb, int nseg, bool vec, int cus) {
  // the kernel needs one whole 16-byte load a column, and has 32-bit offsets into the four matrices of a segment
  if (H < 8 || 4LL * ((H + 7) / 8 * 8) * ((H + 31) / 32 * 32) >= 1LL << 32) return -1;
  int rounds = 1;
  for (int shape = H > 512 ? 1 : 0; shape < 4; ++shape) {
    const int rows = shape == 0 ? 4 : 8, cols = shape <= 1 ? 16 : (shape == 2 ? 32 : 64);
    const long long wgs = (long long)((H + rows - 1) / rows) * ((mb + cols - 1) / cols);
    if (wgs <= cus && shape < 3) return (shape == 2 && H > 1024 && H % 8 == 0) ? -1 : shape;
    rounds = (int)((wgs + cus - 1) / cus);
  }
  if (H % 8 == 0 && (rounds > 1 || H > 1024)) return -1;
  return rounds * (4.0 + 0.0115 * H * nseg) < zr_fused_node_us(H, mb, nseg, vec, cus) ? 3 : -1;
}

// ---- the output layer's error pass (softmax_error_kernel): columns a workgroup adds up, one after another

// 32 keep the partial sums of the bias gradient small against the matrix.  Fewer where 1024-row blocks of 32 columns would
// leave compute units without a workgroup: V = 1000, 33 columns are two workgroups, whose threads wait for 32 columns in turn
// (the whole backward call 51 us against 41 with one column a workgroup and separate bias sums).
inline int zr_softmax_error_cols(int V, int n) {
  const long long row_blocks = (V + 1023) / 1024;
  int cols = 32;
  while (cols > 2 && row_blocks * ((n + cols - 1) / cols) < 256) cols /= 2;
  return cols;
}
