// One LSTM node (one layer, one time step) on narrow tiles: a workgroup owns ROWS hidden rows -- 4 * ROWS weight rows, all
// four gates -- for one column tile, and its 8 waves split the K range of all segments together.
//
// lstm_fused_kernel (zr_lstm.hip) gives a workgroup 32 rows x 4 gates: a single node of a small model is then a dozen or two
// workgroups whose K loops are many times longer than the weights' way from memory, and dividing K across workgroups as
// well costs a round of partial tiles through memory.  Tiles of 4 or 8 rows put a node on 8 (4) times as many workgroups
// with no exchange between them: one LDS sum of the 8 waves and the cell.
// What bounds it: the weights' way from the memory-side cache at narrow batches (H = 1000, 12 columns: 36 MB in 10.9 us, 3.3 TB/s), the matrix pipe at wide ones.
//
// Inputs are read as they lie (columns of H floats, gathered from the embedding for a bottom layer), four consecutive k a
// lane with one 16-byte load that only needs 4-byte alignment, so any H >= 8 runs here: the last load of a column is moved
// down to end inside it and its values are shifted back before they are used.
#include "zr_internal.h"
#include "zr_math.h"
#include "zr_mfma_core.h"
#include "zr_rules.h"

namespace {

constexpr int kWaves = 8;
constexpr int kRedLd = 36;  // LDS row of 32 partial sums, padded

struct LstmRows {
  const float* W;      // [nseg][4] packed fp32 matrices
  const float* bias;   // [4][H]
  const float* in[3];  // segment inputs, columns of H floats
  const int* ids;      // non-null: column n of segment 0 is in[0] + clamp(ids[n]) * H
  const float* cprev;
  const int* mask01;
  float *h, *c;
  float* gates[4];     // all null or all non-null
  float* hp;           // optional: h also k-interleaved, [H/4][mb][4]
  int nseg, V, H, mb, ldw, kp, j_tiles, n_tiles;
  float clip;
};

typedef zr_f32x4 zr_f32x4_u __attribute__((aligned(4)));

// NARROW: 16 columns on the 16 x 16 x 4 instruction; else TN tiles of 32 columns on the 32 x 32 x 2 one (ROWS = 8).
// PF: k-groups in flight.
template <int ROWS, int TN, bool NARROW, int PF>
__global__ void __launch_bounds__(64 * kWaves, 2) lstm_rows_kernel(LstmRows P) {
  static_assert(NARROW ? TN == 1 : ROWS == 8, "tile shape");
  constexpr int KB = NARROW ? 4 : 2;            // k-blocks of 4 per k-group
  constexpr int NB = NARROW ? ROWS / 4 : 1;     // weight sub-tiles
  constexpr int COLS = NARROW ? 16 : 32 * TN;
  constexpr int NOUT = (ROWS * COLS + 511) / 512;
  constexpr int NS = PF + 1;
  __shared__ float red[kWaves * COLS * kRedLd];
  // Workgroup ids congruent mod 8 share a die: the column tiles of a row tile, which read the same weights, go together, and so do two row tiles of
  // four, whose rows are the halves of the weights' 128-byte lines (apart, every line is fetched by two dies: a node of H = 1000 at 12 columns 14.3 us
  // against 10.9, of H = 500 7.2 against 7.0).
  constexpr int RT = ROWS == 4 ? 2 : 1;
  const int id = blockIdx.x, slots = RT * P.n_tiles, at = (id >> 3) % slots;
  const int jt = ((id / (8 * slots)) * 8 + (id & 7)) * RT + at % RT;
  const int nt = at / RT;
  if (jt >= P.j_tiles) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int kslice = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = P.H, mb = P.mb;
  const int j0 = jt * ROWS;
  const int n0 = nt * COLS;
  const int cl = NARROW ? (lane & 15) : (lane & 31);
  const int kq = NARROW ? (lane >> 4) : (lane >> 5);

  // the outputs this thread finishes; their operands are fetched ahead of the K loop
  int oj[NOUT], on[NOUT];
  bool ok[NOUT];
  float bi[NOUT], bf[NOUT], bc[NOUT], bo[NOUT], cprev_v[NOUT], mask_v[NOUT];
#pragma unroll
  for (int u = 0; u < NOUT; ++u) {
    const int o = tid + 512 * u;
    oj[u] = o % ROWS;
    on[u] = o / ROWS;
    const int j = j0 + oj[u], n = n0 + on[u];
    ok[u] = o < ROWS * COLS && n < mb && j < H;
    const int jc = j < H ? j : H - 1, nc = n < mb ? n : mb - 1;
    bi[u] = P.bias[jc], bf[u] = P.bias[H + jc], bc[u] = P.bias[2 * H + jc], bo[u] = P.bias[3 * H + jc];
    cprev_v[u] = P.cprev[(long long)nc * H + jc];
    mask_v[u] = (float)P.mask01[nc];
  }

  // this lane's columns and weight rows
  long long col_off[TN], col_off0[TN];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
    int c = n0 + tn * 32 + cl;
    c = c < mb ? c : mb - 1;
    col_off[tn] = (long long)c * H;
    col_off0[tn] = col_off[tn];
    if (P.ids) {
      const int v = P.ids[c];
      col_off0[tn] = (long long)(v < 0 ? 0 : (v >= P.V ? P.V - 1 : v)) * H;
    }
  }
  const long long HH = (long long)P.kp * P.ldw;
  unsigned woff[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int c = cl + 16 * b;
    woff[b] = (unsigned)((c / ROWS) * HH + 4 * (j0 + c % ROWS));
  }
  const int G = (P.kp + 4 * KB - 1) / (4 * KB);  // k-groups per segment
  const int total = P.nseg * G;
  const int kb_max = (P.kp >> 2) - 1;

  struct Frag {
    zr_f32x4 w[NB], x[TN];
  };
  Frag f[NS];
  // The k-groups of all segments in one row, dealt to the waves in turn: group r is (segment r / G, group r % G).
  int ls = kslice / G, lg = kslice - ls * G, lr = kslice;  // the next group to load
  auto load = [&](Frag& q) {
    const float* Ws = P.W + 4 * HH * ls;
    const int kb = KB * lg + kq;
    const int kbc = NARROW && kb > kb_max ? kb_max : kb;  // (a narrow group may be half: made zero before it is multiplied)
#pragma unroll
    for (int b = 0; b < NB; ++b) q.w[b] = *(const zr_f32x4*)(Ws + (woff[b] + (unsigned)(kbc * 4 * P.ldw)));
    const int k0 = 4 * kb;
    const int ks = k0 < H - 4 ? k0 : H - 4;
    const float* xs = P.in[ls];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) q.x[tn] = *(const zr_f32x4_u*)(xs + ((ls == 0 ? col_off0[tn] : col_off[tn]) + ks));
    // past the end: the last group again (not multiplied)
    if (lr + kWaves < total) {
      lr += kWaves;
      lg += kWaves;
      while (lg >= G) lg -= G, ++ls;
    }
  };
  typedef float acc16 __attribute__((ext_vector_type(16)));
  // Several accumulators, for k of one remainder each: a chain of additions rounds the less the shorter it is, and the older
  // kernels divide K further.  Error of h against 64 bits at H = 1024, one column 2.6e-7 with one accumulator, 1.7e-7 with four
  // (K split across workgroups 1.7e-7), with feed-input 3.3e-7, 1.9e-7 (1.9e-7); H = 500 at 128 columns 2.0e-7, 1.6e-7 with
  // two (1.6e-7).  Costs 0 to 1.5 %.
  constexpr int NACC = NARROW ? 4 : 2;
  acc16 acc[2][TN];
  zr_f32x4 acc4[NACC][NB];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][tn][r] = acc[1][tn][r] = 0.0f;
#pragma unroll
  for (int e = 0; e < NACC; ++e)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc4[e][b] = {0.0f, 0.0f, 0.0f, 0.0f};
  int mg = kslice % G;  // the group (inside its segment) multiplied next
  auto mma = [&](Frag& q) {
    if (4 * KB * (mg + 1) > H) {  // the column ends inside this group: shift the moved loads back, zero what lies behind
      const int k0 = 4 * (KB * mg + kq);
      if (NARROW && KB * mg + kq > kb_max) {  // (both operands: zero times an infinite weight is not zero)
#pragma unroll
        for (int b = 0; b < NB; ++b) q.w[b] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      const int d = k0 < H - 4 ? 0 : k0 - (H - 4);
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const zr_f32x4 v = q.x[tn];
        q.x[tn][0] = d == 0 ? v[0] : (d == 1 ? v[1] : (d == 2 ? v[2] : (d == 3 ? v[3] : 0.0f)));
        q.x[tn][1] = d == 0 ? v[1] : (d == 1 ? v[2] : (d == 2 ? v[3] : 0.0f));
        q.x[tn][2] = d == 0 ? v[2] : (d == 1 ? v[3] : 0.0f);
        q.x[tn][3] = d == 0 ? v[3] : 0.0f;
      }
    }
    mg += kWaves;
    while (mg >= G) mg -= G;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (NARROW) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          zr_f32x4& a = acc4[e & (NACC - 1)][b];
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(q.x[0][e], q.w[b][e], a, 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          acc[e & 1][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(q.x[tn][e], q.w[0][e], acc[e & 1][tn], 0, 0, 0);
      }
    }
  };
  if (kslice < total) {
    const int n_mine = (total - kslice + kWaves - 1) / kWaves;
#pragma unroll
    for (int s = 0; s < PF; ++s) load(f[s]);
    int it = 0;
    for (; it + NS <= n_mine; it += NS) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        load(f[(s + PF) % NS]);
        mma(f[s]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < PF; ++s)
      if (it + s < n_mine) mma(f[s]);
  }

  // partial sums of the K slices through LDS, then the cell
  float* mine = red + kslice * (COLS * kRedLd);
  if constexpr (NARROW) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) mine[(4 * kq + r) * kRedLd + cl + 16 * b] =
            NACC == 4 ? (acc4[0][b][r] + acc4[1][b][r]) + (acc4[NACC - 2][b][r] + acc4[NACC - 1][b][r]) : acc4[0][b][r] + acc4[1][b][r];
  } else {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(tn * 32 + 8 * (r >> 2) + 4 * kq + (r & 3)) * kRedLd + cl] = acc[0][tn][r] + acc[1][tn][r];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NOUT; ++u) {
    if (!ok[u]) continue;
    float z[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float* p = red + on[u] * kRedLd + g * ROWS + oj[u];
      float part[kWaves];
#pragma unroll
      for (int q = 0; q < kWaves; ++q) part[q] = p[q * (COLS * kRedLd)];
      z[g] = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    }
    float gi, gf, gc, go, c, h;
    zr_lstm_cell(z[0] + bi[u], z[1] + bf[u], z[2] + bc[u], z[3] + bo[u], cprev_v[u], mask_v[u], P.clip, gi, gf, gc, go, c, h);
    const int j = j0 + oj[u], n = n0 + on[u];
    const long long ix = (long long)n * H + j;
    P.c[ix] = c;
    P.h[ix] = h;
    if (P.hp) P.hp[((long long)(j >> 2) * mb + n) * 4 + (j & 3)] = h;
    if (P.gates[0]) P.gates[0][ix] = gi, P.gates[1][ix] = gf, P.gates[2][ix] = gc, P.gates[3][ix] = go;
  }
}

}  // namespace

int zr_lstm_rows_step(zr_ctx* ctx, const zr_lstm_weights* w, int nseg, const float* const in[3], const int* d_gather_ids,
                      int V, const float* d_cprev, const int* d_mask01, float clip, int mb, float* d_h, float* d_c,
                      float* const d_gates[4], float* d_hp, int shape) {
  LstmRows P = {};
  P.W = (const float*)w->d_W;
  P.bias = w->d_bias;
  for (int s = 0; s < nseg; ++s) P.in[s] = in[s];
  P.ids = d_gather_ids;
  P.cprev = d_cprev;
  P.mask01 = d_mask01;
  P.h = d_h;
  P.c = d_c;
  for (int g = 0; g < 4; ++g) P.gates[g] = d_gates ? d_gates[g] : nullptr;
  P.hp = d_hp;
  P.nseg = nseg;
  P.V = V;
  P.H = w->H;
  P.mb = mb;
  P.ldw = w->ldw;
  P.kp = w->kp;
  P.clip = clip;
  if (shape == 1 && zr_lstm_rows_halves(P.H, mb, ctx->cu_count)) shape = 0;
  const int rows = shape == 0 ? 4 : 8, cols = shape <= 1 ? 16 : (shape == 2 ? 32 : 64);
  P.j_tiles = (P.H + rows - 1) / rows;
  P.n_tiles = (mb + cols - 1) / cols;
  const int rt = rows == 4 ? 2 : 1;  // row tiles side by side on a die
  const unsigned grid = (unsigned)(((P.j_tiles + rt - 1) / rt + 7) / 8 * 8 * rt * P.n_tiles);
  if (shape == 0)
    lstm_rows_kernel<4, 1, true, 8><<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  else if (shape == 1)
    lstm_rows_kernel<8, 1, true, 8><<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  // 8 x 32 tiles: all of a wave's k-groups in flight at once where ten are enough; else eight, for 128 registers a thread and so two
  // workgroups on a compute unit (160 columns of H = 400 are 280 workgroups with those that leave at once: 15.8 us with ten,
  // 13.3; 128 columns of H = 500 10.3, 9.6; but 128 of H = 300, ten groups a wave, 7.2, 8.1).
  else if (shape == 2 && P.nseg * ((P.kp + 7) / 8) <= 10 * kWaves)
    lstm_rows_kernel<8, 1, false, 10><<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  else if (shape == 2)
    lstm_rows_kernel<8, 1, false, 8><<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  else
    lstm_rows_kernel<8, 2, false, 8><<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("lstm_rows_kernel");
  return ZR_OK;
}
