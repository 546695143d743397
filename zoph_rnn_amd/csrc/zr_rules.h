// Which kernel a call takes, as plain C++ (no device code), so that a rule can be checked without a device against what was
// measured on both sides of its line (tests/test_rules_cpu.py holds the measurements).
#pragma once

// ---- one LSTM node: tiles of 4 or 8 hidden rows (zr_lstm_rows.hip) or launch_fused (zr_lstm.hip)

// launch_fused's time for `units` independent fp32 nodes in one launch, us.  vec: H % 4 == 0 and 16-byte aligned inputs.  Follows
// its own choice of kernel; the constants are fitted to H = 64 .. 2000 at 1 .. 512 columns, one node with two and three segments
// and up to four nodes with two, and hold to about 10 % (H below 200: 20 %).  No launch beats its weights at 7 TB/s.
inline double zr_fused_us(int units, int H, int mb, int nseg, bool vec, int cus) {
  const int j = units * ((H + 31) / 32), n32 = (mb + 31) / 32;
  const int whole = j * ((n32 + 1) / 2);
  const double weights = 6.0 + 16.0 * units * nseg * H * H / 7.0e6;
  double us;
  if (H % 8 == 0 && vec && whole < 200) {
    const int tiles = j * n32;
    int parts = (cus + tiles / 2) / tiles;
    if (parts > H / 128) parts = H / 128;
    if (parts > 8) parts = 8;
    if (parts >= 2) {  // K split across workgroups; the row tiles are dealt to the eight dies
      const int rounds = ((j + 7) / 8 * n32 * parts + cus / 8 - 1) / (cus / 8);
      us = rounds * (6.5 + 0.8 * parts + 0.018 * H / parts * nseg);
      return us > weights ? us : weights;
    }
  } else if (vec && n32 >= 3 && whole < 200) {  // weights through LDS
    const int tiles = j * ((n32 + 3) / 4);
    int parts = cus / (tiles * nseg);
    if (parts > 8) parts = 8;
    if (parts > (H + 31) / 32) parts = (H + 31) / 32;
    if (parts < 1) parts = 1;
    const int rounds = (tiles * nseg * parts + cus - 1) / cus;
    us = rounds * (12.5 + 0.075 * H / parts + 3.0 * parts);
    return us > weights ? us : weights;
  }
  const bool fast = H % 8 == 0 && vec;  // whole k-groups, wide loads
  const int tn = n32 >= 2 && whole > 128 ? 2 : 1;
  const int wgs = j * ((n32 + tn - 1) / tn);
  if (wgs < 192)
    us = 6.0 + (fast ? (tn == 2 ? 0.014 : 0.0165) : (vec ? 0.026 : 0.030)) * H * nseg * tn;
  else
    us = (wgs + cus - 1) / cus * (6.5 + (tn == 2 ? (fast ? 0.0295 : 0.036) : (fast ? 0.0165 : 0.0205)) * H * nseg);
  return us > weights ? us : weights;
}

// Tile by size, one node of H = 1000 / 500 / 300 at up to 128 columns, us (the register-streaming kernel of zr_lstm.hip
// with K split across workgroups: 16-27 / 30-33 / 23-30):
//   4 x 16:  10.9 at 12 columns /  7.0 at 12, 9.6 at 37 /  5.4 at 20      8 x 16:  12.7 at 12, 12.0 at 32 / 8.2 at 37 / 6.4
//   8 x 32:  17.0 at 64 / 11.7 at 128 / 7.7 at 100                        8 x 64:  26.5 at 128 / 16.8 at 128
// The smallest tile that keeps the workgroups within one per compute unit wins (4 x 16 beyond H = 512: zr_lstm_rows_halves).  Wide tiles of a long K range lose to the streaming kernel where that has
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
  return rounds * (4.0 + 0.0115 * H * nseg) < zr_fused_us(1, H, mb, nseg, vec, cus) ? 3 : -1;
}

// 8 x 16 tiles as twice as many of 4 x 16, whose two halves of a line go to the same die, while those are within one a compute unit: us of a node, 8 x 16 / 4 x 16, 16
// columns, H = 513 8.9 / 7.7, 600 10.1 / 8.9, 800 11.4 / 10.0, 1000 12.9 / 11.2, 1024 12.6 / 11.0; one column, 1000 11.9 / 10.6.
inline bool zr_lstm_rows_halves(int H, int mb, int cus) { return (long long)((H + 3) / 4) * ((mb + 15) / 16) <= cus; }

// The same for a node on bf16 weights (zr_lstm_rows_bf16.hip against lstm_fused_kernel's 32-row tiles); shapes 1 to 3 as above.  us of a
// node, two terms (one term), in a decoder step of four layers: H = 512, 64 columns 12.1 -> 6.2 on 8 x 32 tiles (10.7 -> 5.2), 1024, 12
// columns 15.4 -> 7.9 (14.2 -> 7.1), 1024, 64 17.3 -> 9.6, 1024, 128 17.2 -> 13.7 on 8 x 64, 2000, 64 35.0 -> 30.0.  Any of the tiles wins while its
// workgroups are within one a compute unit, the narrowest the most; 8 x 16 against 8 x 32 only where it fills more of the chip (1024, 32 columns
// 8.1 / 9.5; 512, 37 6.1 / 6.0).  In a second round the activations, which every row tile reads, are too much: 1024, 192 columns 17.5 against
// 21.6 and 24.0, 768, 192 14.3 / 18.2; but for three 32-column tiles where 64-column ones are two rounds as well, 1104, 80 columns 16.4 / 14.2.
inline int zr_lstm_rows_bf16_shape(int H, int mb, int cus) {
  const long long rows = H / 8;
  if (4LL * H * ((H + 31) / 32 * 32) >= 1LL << 31 || 8LL * H * mb >= 1LL << 31) return -1;  // 32-bit offsets
  if (H > 512 && mb > 16 && rows * ((mb + 15) / 16) <= cus) return 1;
  if (rows * ((mb + 31) / 32) <= cus) return 2;
  if (rows * ((mb + 63) / 64) <= cus) return 3;
  return mb > 64 && mb <= 96 && 4 * rows * 3 <= 7LL * cus ? 2 : -1;
}

// ---- the sweep of a stack (zr_lstm_stack_forward): one launch per diagonal, one launch with streamed weights
// (lstm_sweep_kernel), or with its weights in registers (lstm_resident_kernel).  Estimates in us; the least one is taken.
// Against 1812 sizes (H = 64 .. 2000, 1 to 4 layers, 1 to 256 columns, 12 and 50 steps; all that fit measured for each) the
// choice is 0.2 % from the best schedule on average, more than 10 % for about one size in a hundred.

// One launch per diagonal: the first and last few have fewer layers than the others.
inline double zr_sweep_diagonals_us(int nl, int H, int mb, int T, bool vec, int cus) {
  const int full = nl < T ? nl : T;
  double us = (T + nl - 1 - 2 * (full - 1)) * zr_fused_us(full, H, mb, 2, vec, cus);
  for (int units = 1; units < full; ++units) us += 2.0 * zr_fused_us(units, H, mb, 2, vec, cus);
  return us;
}

// Streamed weights on tiles of 32 * tn columns: a hand-over, a little more with every layer, and the steps of 64 k of both segments (an even number of
// each) at 0.74 us of 32 columns and 1.18 of 64, or the weights at 6 TB/s where they outgrow the caches (4 layers of H = 2000 85 us a
// step); half a step more per layer to fill.  Within 17 % of 297 sizes (H = 128 .. 2000, 12 to 256 columns), 4 % on average.
inline double zr_sweep_streamed_us(int nl, int H, int T, int tn) {
  const double steps = (H + 127) / 128 * 4.0, weights = 32.0 * nl * H * H / 6.0e6 + 3.5;
  const double k_loop = tn == 1 ? 3.6 + 0.42 * nl + 0.74 * steps : 1.5 + 1.6 * nl + 1.18 * steps;
  return (T + 0.5 * nl) * (k_loop > weights ? k_loop : weights);
}

// Resident weights, one launch of `layers` layers (the sweep's first or a later one): classes by H up to 128, 256, 512, 1024 and
// by 16, 32, 64 columns a workgroup.  A time step takes what its class takes -- every workgroup has the registers, and walks
// the k-groups, of the largest H of the class -- as long as each compute unit has one workgroup (H = 500: 4.1 us at 16 to 64
// columns on 16-column tiles, 7.2-7.5 at 16 to 128 columns on 32-column tiles).  Later launches read h and no embedding.  With
// two workgroups on some compute units a step takes about that much longer and the two get in each other's way (H = 500, 504
// workgroups: 11.1), less so when they belong to different layers.  Filling the registers costs a few us a layer.
inline double zr_sweep_resident_us(int size_class, int col_class, bool first, int layers, long long wgs, int T, int cus) {
  const double step_first[4][3] = {{2.45, 3.1, 4.6}, {3.05, 4.15, 8.6}, {4.15, 6.9, 15.0}, {6.3, 11.5, 0.0}};
  const double step_later[4][3] = {{2.4, 3.0, 4.6}, {3.0, 4.1, 6.7}, {4.1, 6.0, 11.0}, {6.0, 10.4, 0.0}};
  const double two[3][2] = {{1.0, 1.0}, {1.4, 0.6}, {1.8, 0.5}}, two_wide[3][2] = {{1.3, 0.6}, {1.7, 0.3}, {1.7, 0.3}};
  const double fill[4] = {1.0, 2.5, 4.5, 9.0};
  double step = (first ? step_first : step_later)[size_class][col_class];
  if (wgs > cus && size_class < 3) {
    const double* f = (col_class ? two_wide : two)[size_class];
    step *= f[0] + f[1] * ((double)wgs / cus - 1.0) - (col_class == 0 && size_class == 2 && layers > 1 ? 0.35 : 0.0);
  }
  return (T + layers - 1) * step + 6.0 + fill[size_class] * layers;
}

// Column class and layers a launch: the cheapest of those that fit.  capacity: workgroups of each column class the device holds
// at once (0: no such kernel); flags: hand-over flags there are.  us < 0: none fits.
constexpr int kResidentColumns[3] = {16, 32, 64};
struct ZrResidentPlan {
  int size_class, col_class, n_tiles, at_once, flag_stride;
  double us;
};
inline ZrResidentPlan zr_sweep_resident_plan(int nl, int H, int mb, int T, const int capacity[3], int flags, int cus) {
  ZrResidentPlan plan = {H <= 128 ? 0 : (H <= 256 ? 1 : (H <= 512 ? 2 : 3)), 0, 0, 0, 0, -1.0};
  const int row_tiles = (H + 7) / 8;
  const int producers = 2 << plan.size_class;  // of a wave's K slice, in every column class
  plan.flag_stride = (8 * producers + 31) / 32 * 32;
  for (int c = 0; c < 3; ++c) {
    const int n_tiles = (mb + kResidentColumns[c] - 1) / kResidentColumns[c];
    int at_once = capacity[c] / (row_tiles * n_tiles);
    if (at_once > nl) at_once = nl;
    while (at_once > 0 && (long long)at_once * n_tiles * plan.flag_stride > flags) --at_once;
    if (at_once < 1) continue;
    double us = 0.0;
    for (int l = 0; l < nl; l += at_once) {
      const int now = nl - l < at_once ? nl - l : at_once;
      us += zr_sweep_resident_us(plan.size_class, c, l == 0, now, (long long)now * row_tiles * n_tiles, T, cus);
    }
    if (plan.us < 0.0 || us < plan.us) plan.us = us, plan.col_class = c, plan.n_tiles = n_tiles, plan.at_once = at_once;
  }
  return plan;
}

// ---- the backward sweep of a stack: a launch or two per diagonal, or one launch with its weights in registers
// (lstm_backward_resident_kernel)

// Where a layer's workgroups of 16 rows x 16 columns fit the device they win with up to four launches, at 24 steps, us per diagonal / in
// registers: 2 x 100, 100 columns 225 / 106, 3 x 200, 64 307 / 136, 4 x 200, 128 (two launches) 403 / 282, 2 x 500, 64 405 / 230, 3 x 500, 128 (three) 799 /
// 564, 4 x 500, 128 (four) 850 / 752; but with eight, 8 x 300, 128 821 / 1099, 8 x 500, 128 1219 / 1536: the layers no longer overlap.
// Sizes share a kernel by their k-groups a wave; the one for 257 to 320 against the next larger one: 2 x 300, 20 columns, 35 steps 207 / 221, 3 x 320, 64 182 / 194, 1 x 257, 20 112 /
// 117.
constexpr int kBackLaunches = 4;
constexpr int ZR_BACK_CLASSES = 5;
inline int zr_back_size_class(int H) { return H <= 128 ? 0 : (H <= 256 ? 1 : (H <= 320 ? 2 : (H <= 384 ? 3 : 4))); }
struct ZrBackPlan {
  int size_class, at_once, flag_stride;  // layers a launch; 0: it does not fit
  bool below;                            // the last launch also makes the error to the input from below
  int capacity;                          // workgroups the device holds at once
};
// capacity: workgroups the device holds at once; below: whether the caller wants the error to the input from below.
inline ZrBackPlan zr_back_plan(int nl, int H, int mb, int T, bool below, int capacity, int flags) {
  ZrBackPlan plan = {zr_back_size_class(H), 0, 0, false, capacity};
  const int tiles = (H + 15) / 16, n_tiles = (mb + 15) / 16;
  plan.flag_stride = (tiles + 31) / 32 * 32;
  const long long per = (long long)tiles * n_tiles;
  long long fit = capacity / per;
  if (fit > nl) fit = nl;
  while (fit > 0 && fit * n_tiles * plan.flag_stride > flags) --fit;
  if (fit < 1) return plan;
  plan.at_once = (int)fit;
  const int last = nl % plan.at_once ? nl % plan.at_once : plan.at_once;
  plan.below = below && (last + 1) * per <= capacity;
  return plan;
}

inline bool zr_back_takes(const ZrBackPlan& plan, int nl) { return plan.at_once > 0 && (nl + plan.at_once - 1) / plan.at_once <= kBackLaunches; }

// ---- normalising the output matrix (softmax_normalize_kernel): 16-byte accesses a thread, and whether its workgroups fold the block pairs

// Every workgroup folds its column's V / 32 pairs: cheaper than a launch for it until there are some 1.25 million to fold (counted for four accesses a
// thread), 2.2 million up to 32768 rows, a few pairs a thread.  us behind the product, folding with two accesses a thread / with four / in a launch of its own: 50000 x 48 (0.98)
// 10.5 / 10.8 / 11.0, 40000 x 96 (1.2) 13.8 / 14.1 / 13.3, 50000 x 64 (1.3) 12.7 / 13.4 / 12.5, 80000 x 64 (3.2) 15.1 / 14.9 / 13.6; 30000 x 128 (0.96) 14.2 / 10.2 / 13.6,
// 20000 x 600 (1.9) 22.1 / 19.0 / 21.0, 30001 x 384 (2.9) 20.5 / 20.4 / 19.0.  Two accesses where there is little to fold, 50000 x 1 3.7 / 4.2; four where columns start
// at odd addresses: 30011 x 37 6.7 / 5.7.
struct ZrNormalizePlan {
  int accesses;
  bool fold;
};
inline ZrNormalizePlan zr_softmax_normalize_plan(int V, int n) {
  const double folds = (double)((V + 4095) / 4096) * n * ((V + 31) / 32);
  if (folds > (V <= 32768 ? 2.2e6 : 1.25e6)) return {2, false};
  return {V <= 1024 ? 1 : (V % 4 || folds > 0.9e6 ? 4 : 2), true};
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

// ---- large fp32 products: the split product (zr_split_gemm.hip) or the fp32 kernels

// Estimated microseconds of a split product's launch of `wgs` workgroups of `steps` steps of 32 k each, on tiles of 128 rows x
// 64 * tnw columns.  A step of one workgroup alone on its compute unit, of two, of three sharing it (measured; 128-column
// tiles hold three, 256-column tiles two).
inline double zr_split_launch_us(int tnw, long long wgs, int steps, int cus) {
  const double us128[4] = {0.0, 2.8, 3.7, 5.0}, us256[3] = {0.0, 3.7, 5.8};
  const int cap = tnw == 4 ? 2 : 3;
  const double* us = tnw == 4 ? us256 : us128;
  const long long per_cu = (wgs + cus - 1) / cus;
  return ((double)(per_cu / cap) * us[cap] + us[per_cu % cap]) * (steps + 1.5);
}

// Against the fp32 kernels (both with their launches' own preparation, us): 10001 x 300 x 700 63 / 97, 300 x 700 x 10001
// 62 / 101, 4000 x 1000 x 6400 312 / 472, 33333 x 700 x 500 174 / 327; but 1000 x 128 x 4000 40 / 40 and 1200 x 300 x
// 700 30 / 20: up to 10^9 multiply-adds, or with an output that fills few tiles, there is too little to win.
inline bool zr_split_gemm_takes(int M, int N, int K) {
  return M >= 256 && N >= 256 && K >= 256 && (double)M * N * K > 1.0e9;
}

// The same for a product as zr_gemm_launch has it, whose other choice is one launch without transposes.  Two places where
// the line above lies too low:
//   * Outputs of one to four 32 x 32 blocks a compute unit, row-major operands (M < 2048: beyond that the fp32 choice is
//     another kernel): one wave per block leaves little idle there.  512 x 512 x 4096 37 / 31, 1000 x 1000 x 1000 41 / 34,
//     1001 x 1001 x 1003 42 / 36, 1000 x 1000 x 1100 38 / 38; against it 1500 x 1500 x 500 40 / 64, 300 x 300 x 12000 51 / 89.
//   * The logits with their block statistics, which cannot divide K: a few tiles then walk all of it.  The fp32 kernels
//     reach half of 95 TFLOP/s or more.  2000 x 512 x 1000 (64 tiles) 82-92 / 38-42, 2000 x 1024 x 1000 (128) 96 / 64, 5000 x
//     400 x 500 (160) 56 / 42; 5000 x 512 x 500 (160) 57 / 79, 2000 x 1100 x 1000 (144) 98 / 131.
inline bool zr_split_gemm_takes_product(int M, int N, int K, bool k_fast_a, bool statistics, int cus) {
  if (!zr_split_gemm_takes(M, N, K)) return false;
  const double macs = (double)M * N * K;
  if (statistics) {
    const long long m_tiles = (M + 127) / 128;
    const double narrow = zr_split_launch_us(2, m_tiles * ((N + 127) / 128), (K + 31) / 32, cus);
    const double wide = zr_split_launch_us(4, m_tiles * ((N + 255) / 256), (K + 31) / 32, cus);
    return (narrow < wide ? narrow : wide) <= 2.1 * macs * 2.0 / 95.0e6;
  }
  const long long blocks = (long long)((M + 31) / 32) * ((N + 31) / 32);
  return k_fast_a || M >= 2048 || blocks < cus || blocks > 4 * cus || macs >= 1.1e9;
}

// ---- weight gradients of a single node (outer_accumulate_kernel), `count` products a launch, K = the minibatch

// Against a transpose and the LDS-tiled product each, us of the whole call.  Two H x H at a time (zr_attn_backward): faster at
// every size up to 256 columns, a third over all; all four of a node in one launch, us of its whole backward pass against those: H = 64, 8 columns 33 / 52, 256 46 / 59; 500, 64
// columns 48 / 75; 1000, 256 columns 127 / 172.  One 4H x H (zr_lstm_feed_backward): H = 1000, 128 columns 63 / 82, 200
// 75 / 89; but small ones do not fill the chip with waves that each walk all columns: H = 64, 192 columns 20.8 / 19.1, 256
// 23.2 / 19.5, H = 256, 192 columns 27.3 / 25.2, where 64 columns are 16.1 / 17.0 and 22.9 / 23.9.
inline bool zr_outer_takes(int count, int M, int N, int K) {
  return K <= (count > 1 || (long long)M * N >= 300000 ? 256 : 96) && !zr_split_gemm_takes(M, N, K);
}

// ---- weight gradients of a layer over N columns: one launch in fp32 (weight_gradients_kernel), or transposes and products (on the bf16 matrix cores
// where the split product takes them) and row sums

// us, those / this one (steps x minibatch): H = 64, 20 x 8 20 / 9, 100, 20 x 20 21 / 14, 300, 35 x 20 40 / 21, 500, 24 x 64 99 / 78, 700, 20 x 20 94 / 55; but few tiles that each
// walk many columns, 64, 50 x 64 40 / 76, 200, 50 x 64 69 / 79, and what the bf16 matrix cores do faster, 500, 60 x 128 262 / 367, 1000, 12 x 64 136 / 162.
// Estimates of both, within 10 % here and 30 % there.
inline bool zr_weight_gradients_takes(int H, long long N, int cus) {
  const long long tiles = (4LL * H + 63) / 64 * ((H + 63) / 64) * 2;
  const double gflop = 16.0e-9 * H * H * N;
  const double here = 4.0 + (double)((tiles + cus - 1) / cus) * (2.5 + 0.0235 * N);
  const double there = 20.0 + gflop / 0.13 + (gflop < 2.5 ? 10.0 * gflop : 25.0);
  return here <= 0.9 * there;
}

// ---- grouped products (the error products of a diagonal of the backward sweep, K = 4H): `tiles` of 32 x 32 with K over eight
// waves, or 64 x 64 tiles (64 x 32 up to 32 columns)

// Up to one such workgroup a compute unit the small tiles take half the time or less: whole sweeps of 20-24 steps, 80 tiles a
// full diagonal (2 x 300, 64 columns) 682 -> 351 us, 128 (2 x 500, 64) 1156 -> 540, 256 (2 x 1000, 64) 1662 -> 721.  With up to
// one and a half, in two rounds, a sweep is 9 to 13 % faster than on 64 x 64 tiles (2 x 768, 128 columns, 12 steps 789 -> 701;
// 3 x 300, 192 columns 474 -> 482 the one exception of 37) -- but not up to 32 columns, where the larger tiles leave no more
// idle (4 x 1200, 32 columns 746 -> 989).  Up to two workgroups a compute unit it goes either way: 2 x 1000, 128 columns
// 970 -> 884, 4 x 500, 128 columns 665 -> 588, but 2 x 600, 192 columns 719 -> 804 and 4 x 300, 192 columns 531 -> 571, without
// a size that tells them apart; beyond that it loses (3 x 1000, 128 columns 1098 -> 1317).
inline bool zr_grouped_small_tiles(long long tiles, int columns, int cus) {
  return tiles <= cus || (columns > 32 && 2 * tiles <= 3LL * cus);
}

// The same products on k-interleaved operands as three bf16 terms, 64 x 64 tiles (zr_error_products.hip): faster as soon as there are more 32 x 32
// tiles than compute units, beyond 32 columns.  us of a sweep of 12 steps on the kernels above / on this one: 4 x 300, 100 columns (320 tiles)
// 388 / 343, 1 x 768, 192 columns (288) 626 / 505, 4 x 1000, 128 columns (1024) 1190 / 922, 2 x 1200, 192 columns (912) 3041 / 912; but 2 x
// 500, 128 columns (256) 313 / 411, and 4 x 2000, 20 columns (504) 1499 / 1546.
inline bool zr_error_products_takes(long long tiles, int columns, int cus) { return tiles > cus && columns > 32; }

// ---- small products (zr_small_gemm.hip): narrow tiles whose waves have all their operands in flight

// Shape: 0 = 16 rows x 16 columns, 1 = 16 x 32, 2 = 32 x 32, -1 = the other kernels.  z: independent products of one launch.  a_pack,
// trans_a: the left operand's layout as ZrGemmDesc has it.  Estimates of a launch in us: a trip to memory and the launch, and the K range of a
// workgroup, alone on its compute unit or beside a second one; beyond two a compute unit the wider tiles of the other kernels win, and so they do
// where 32 x 32 tiles are the best choice here and the matrix is read 4 bytes a lane (column-major), or row-major up to K = 1500: 1000 x 256 x 1000
// 11.8 / 10.2 and 11.4 / 10.8; and on column-major matrices beyond one and three quarters: 1111 x 110 x 736 8.6 / 8.0.
// This one / the others, us: 500 x 64 x 500 4.2 / 7.0 column-major; 1000 x 64 x 1000 6.2 / 9.5; 2 products of 500 x 128 x 2000 13.7 / 16.8, 1000 x 20 x
// 4000 14.9 / 27.3; 100 x 20 x 100 row-major 3.2 / 4.1; an attention step on prepared matrices, H = 500, 37 columns 19.6 / 35.2; bf16 matrices, H = 1024,
// 64 columns 24.0 / 30.4; sweeps back through 12 steps, 2 x 100, 128 columns 136 / 242, 2 x 500, 64 columns 243 / 293, 2 x 1000, 128 columns 771 /
// 966.  Of 485 sizes of one and two products the choice is 1.7 % from the best shape on average, and slower than the others at two: 819 x 143 x 1176
// row-major 13.2 / 11.4, 1156 x 193 x 20 4.1 / 3.9.
inline int zr_small_gemm_shape(int M, int N, int K, int nseg, int z, int a_pack, bool trans_a, int cus) {
  if (K < 16) return -1;
  const double slope[3] = {0.0036, 0.0052, 0.0078}, second[3] = {1.55, 1.8, 1.9};
  const double k = (double)K * nseg * (a_pack == 2 ? 0.5 : 1.0);  // bf16 weights: twice the k for the same bytes and instructions
  int best = -1;
  double us = 0.0;
  for (int s = 0; s < 3; ++s) {
    const int rows = s == 2 ? 32 : 16, cols = s == 0 ? 16 : 32;
    const long long wgs = (long long)((M + rows - 1) / rows) * ((N + cols - 1) / cols) * z;
    if (wgs > 2LL * cus || (s == 0 && a_pack == 0 && !trans_a && 4 * wgs > 7LL * cus)) continue;
    const double t = 3.4 + slope[s] * k * (wgs > cus ? second[s] : 1.0);
    if (best < 0 || t < us) {
      best = s, us = t;
      if (s == 2 && (a_pack == 0 ? !trans_a || k < 1500.0 : a_pack == 2 && wgs > cus && k > 512.0)) best = -1;
    }
  }
  return best;
}

// Groups a wave has in flight: all it has, up to 64 registers of operands.
inline int zr_small_gemm_depth(int shape, int K, int nseg, int a_pack) {
  const int kg = a_pack == 2 ? 32 : 16, mine = (nseg * ((K + kg - 1) / kg) + 7) / 8;
  if (shape == 0) return mine <= 2 ? 2 : (mine <= 4 ? 4 : 8);
  return shape == 1 ? (mine <= 3 ? 3 : 6) : 4;
}

// ---- sums over the columns of an attention node's backward pass (rows_with_sum): workgroups that share the columns of 32 rows

// us of both sums' kernels, an element-wise one and a separate sum / one workgroup that walks all columns / in parts: H = 64, 64 columns 9.6 /
// 5.6, 512 15.4 / 9.9, 1024 15.9 / 15.4 / 13.1, 2048 19.3 / 25.9 / 12.4; H = 1000, 64 14.7 / 6.6, 512 28.2 / 11.9, 1024 28.8 / 23.0 / 20.4, 2048
// 32.0 / 47.2 / 24.9.
inline int zr_attn_sum_parts(int mb) { return mb <= 512 ? 1 : (mb + 255) / 256; }

// ---- the output layer's product on a prepared fp32 matrix (zr_logits.hip)

// tn: 32-column blocks of a tile, waves: 32-row blocks of a workgroup; tn = 0: the other kernels.
// Estimated time, us: (steps of 32 k + what filling and the epilogue take) * a step of the workgroups that share a compute unit (one of four
// waves alone; two of four or one of eight, whose matrix instructions fill it), times the rounds: within 11 % of 2700 measured
// launches (V = 1000 .. 50000, H = 64 .. 1000, 33 to 1000 columns), and the choice is 4 % from the best tile on average.
// Against the kernels before, the product alone, us: 50000 x 128 x 1000 123 -> 89 to 92, 192 columns 173 -> 125 to 133, 30011 x 33 x 500 30 ->
// 21, 33333 x 700 x 500 206 -> 171, 50000 x 128 x 333 79 -> 39, 16000 x 700 x 200 172 -> 53, 1000 x 64 x 64 8.9 -> 5.1.  Beyond 1024 columns the split product on the
// plain matrix keeps what it takes, but for half-empty tiles: it has 256-column tiles and fewer conversions, and the estimate above does not know
// the clock a launch of milliseconds runs at (50000 x 6400 x 1000 3.93 ms there, 4.09 here and 1.4 ms more inside a training
// step; 20000 x 1280 x 500 208 us, 204; but 3000 x 3000 x 1000 171, 126).
// Not where up to three 32 x 32 blocks a compute unit with K over eight waves are all there is to do and K is long: 1000 x 64 x 1000 10.3
// against 24.2, 4000 x 128 x 777 17.3 / 20.5; but 4000 x 192 x 777 24.4 / 20.7, 8000 x 128 x 1000 28.2 / 25.3, 4000 x 192 x 500 18.0 / 14.9.
struct ZrLogitsPlan {
  int tn, waves;
};
inline ZrLogitsPlan zr_logits_plan(int V, int cols, int H, int cus) {
  ZrLogitsPlan plan = {0, 0};
  const long long blocks = (V + 31) / 32, n32 = (cols + 31) / 32;
  // Up to 16 columns: zr_logits_narrow.hip.  Up to 32, us, the other kernels / this one: K % 8 == 0 (a wave of theirs walks all of K on fp32 instructions), 8192 x 256 17.0
  // / 9.0, 20000 x 512 24.4 / 15.1, 50000 x 1000 43.2 / 37.4, 80000 x 512 47.1 / 43.5; otherwise 30011 x 500 20.9 / 17.2, 50000 x 300 27.3 / 15.9, 9000 x 250 8.2 / 9.1; few
  // rows 4000 x 128 8.4 / 6.4, 1000 x 128 6.5 / 6.2, 1000 x 200 7.5 / 8.4, 4000 x 1000 12.0 / 24.5.
  if (cols <= 16 || (cols <= 32 && H > 128 && V < (H % 8 == 0 ? 8192 : 24576))) return plan;
  // 32-bit offsets into the matrix, and a few steps past it
  if ((((long long)H + 7) / 8 * 8 + 160) * blocks * 32 * 4 >= 1LL << 32) return plan;
  const int steps = (H + 31) / 32;
  double best = 0.0;
  for (int tn = 1; tn <= 6; ++tn)
    for (int waves = 8; waves >= 4; waves -= 4) {
      const long long n_tiles = (n32 + tn - 1) / tn, rounds = ((blocks + waves - 1) / waves * n_tiles + cus - 1) / cus;
      const double full = 0.4 + 0.456 * tn, alone = 0.306 + 0.334 * tn;
      // (the matrix is fetched and split once for every column tile)
      const double us = (1.0 + 0.02 * (n_tiles - 1)) * (steps + 3.7) * (waves == 8 ? rounds * full : (double)(rounds / 2) * full + (rounds & 1) * alone);
      if (!plan.tn || us < best) best = us, plan.tn = tn, plan.waves = waves;
    }
  double other = -1.0;
  if (cols > 1024 && zr_split_gemm_takes_product(V, cols, H, false, true, cus)) {
    const long long m = (V + 127) / 128;
    const double narrow = zr_split_launch_us(2, m * ((cols + 127) / 128), steps, cus), wide = zr_split_launch_us(4, m * ((cols + 255) / 256), steps, cus);
    other = (narrow < wide ? narrow : wide) / 1.5;
  } else if (H >= 512 && V < 8192 && blocks * n32 <= 3LL * cus) {
    other = 2.0 + 0.0095 * H * ((blocks * n32 + cus - 1) / cus);
  }
  if (other > 0.0 && other <= best) plan.tn = plan.waves = 0;
  return plan;
}

// The same for up to 16 columns (zr_logits_narrow.hip) instead of 32-column instructions and, below 8192 rows or with K % 8 != 0, the others: faster by 20 to
// 65 % at every size (V = 1000 .. 80000, H = 64 .. 1000) but few rows of a long K, which one wave then walks alone while the others split it over eight from
// K = 512 on: us, those / this one, 4000 x 1000 11.4 / 12.1, 500 x 504 9.2 / 7.6, 500 x 512 6.5 / 7.5, 2040 x 600 7.0 / 8.5, 2050 x 600 8.6 / 8.5, 2050 x 550 6.6 / 8.3, 8000 x 550
// 6.6 / 8.3, 8192 x 777 7.7 / 10.2, 9000 x 550 11.1 / 8.4, 4000 x 200 8.9 / 4.8, 8192 x 300 6.4 / 5.2, 10000 x 1000 37.8 / 12.7.
inline bool zr_logits_narrow_takes(int V, int cols, int H) {
  if (cols > 16 || H < 4) return false;
  if (H >= 512 && (V < 2048 || (H % 8 ? V <= 8192 : V < 8192 && H > 600))) return false;
  return (((long long)H + 7) / 8 * 8 + 160) * (((long long)V + 31) / 32) * 32 * 4 < 1LL << 32;  // 32-bit offsets
}

// Its two forms: workgroups of four waves of 64 rows where they are just about one a compute unit and K is long, else waves of 32 rows.  us of a call
// at 12 columns, the first / the second: 1000 at 44000 rows 29.7 / 29.7, 48000 30.8 / 32.3, 50000 31.6 / 33.4, 56000 34.0 / 36.6, 65536 38.2 / 40.9, 66000 61.2 / 46.2; 512 at 40000 16.2 / 14.8,
// 56000 18.8 / 19.6; 333 at 50000 14.2 / 13.6, 56000 13.4 / 13.5; 200 at 56000 10.5 / 10.0, 65536 11.8 / 10.8; 64 at 50000 4.8 / 4.5.
inline bool zr_logits_narrow_pairs(int V, int H, int cus) {
  const int groups = (V + 255) / 256;
  return H >= 400 && groups <= cus && 10 * groups >= 7 * cus;
}

// The same on a prepared bf16 matrix for up to 64 columns (zr_logits_bf16.hip) instead of gemm_rows_kernel or, up to 32 columns, gemm_kernel, whose workgroups split K over
// their waves: a wave here walks all of K, which few rows pay for.  us of a call, those / this one, 37 columns: 10000 x 512 11.7 / 10.9, 20000 x 1024 18.1 / 16.4,
// 33333 x 512 19.4 / 15.6, 50000 x 64 19.5 / 10.4, 50000 x 1024 34.8 / 27.0, 80000 x 2000 87.4 / 67.5; 8 columns 50000 x 256 10.7 / 8.3, 80000 x 2000 60.4 / 55.1; and
// 8192 x 256 8.5 / 9.2, 8192 x 1024 10.7 / 14.8, 16384 x 1024 13.3 / 15.4, 24000 x 2000 24.7 / 24.2 (8 columns 20.1 / 20.7 the other way).
inline bool zr_logits_bf16_takes(int V, int cols, int H) {
  if (cols > 64 || H % 16 != 0 || V < 10000 || V < 19LL * H) return false;
  return ((long long)H / 8 + 56) * (((long long)V + 31) / 32) * 32 * 16 < 1LL << 32;  // 32-bit offsets, up to seven chunks behind the last one
}

// ---- the clipped update of one matrix (zr_sgd_update): one launch whose workgroups each read the whole gradient, or a launch for the
// norm and one for the update

// us of a call, one launch / two (the second is the time to launch them): 300 values 4.2 / 7.0, 40000 4.2 / 7.0, 90000 5.6 / 7.0, 131072 6.6 / 7.0,
// 160000 7.6 / 7.0, 250000 10.0 / 6.9.  A quarter of that with four bytes a load.
inline bool zr_sgd_small(long long n, bool vec) { return n <= (vec ? 112000 : 28000); }

// One launch whose workgroups exchange their sums (sgd_fused_kernel): 16-byte accesses a thread, 0: not this one.  us, that above / two launches /
// this one with two, four, eight accesses: 28000 4.1 / 7.0 / 4.1, 4.4, 4.8; 90000 6.5 / 6.9 / 4.3, 4.7, 6.0; 250000 - / 7.0 / 4.9, 5.0, 6.3; 500000 - / 7.2 / 5.7, 6.1,
// 7.0; 1000000 - / 8.4 / 6.9, 6.8, 7.9; 2000000 - / 10.2 / -, 8.8, 9.0; 4000000 - / 14.0 / -, -, 11.4.  With one access more workgroups meet: 500000 6.1.
constexpr int kSgdThreads = 1024, kSgdSlots = 128;
inline int zr_sgd_fused_accesses(long long n) {
  constexpr long long most = 4LL * kSgdThreads * kSgdSlots;  // with one access
  return n <= 28000 || n > 8 * most ? 0 : (n <= 2 * most ? 2 : (n <= 4 * most ? 4 : 8));
}
