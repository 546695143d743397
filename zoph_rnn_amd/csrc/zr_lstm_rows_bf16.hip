// One LSTM node on bf16 weights and narrow tiles: the work split of lstm_rows_kernel (zr_lstm_rows.hip) -- a workgroup owns 8 hidden
// rows, 32 weight rows, for one column tile, and its 8 waves split the k-groups of all segments -- on the bf16
// instructions.  Inputs are the bf16 terms that the step has made of every activation once, k-interleaved by 8, so a k-group of an operand is one
// 16-byte load a lane on both sides and needs no conversion.
//
// lstm_fused_kernel's 32-row tiles put a node of H = 1024 at 64 columns on 64 workgroups: 15.8 to 18.1 us, a quarter of the chip
// streaming the weights.  Bound: the weights' way from the memory-side cache, and beyond about 64 columns the activations' from L2, which every row tile
// reads: a node of H = 1024 (nine of 8 MB matrices in four) 7.9 us at 12 columns, 9.6 at 64, 13.7 at 128 with two terms (15.4, 17.3 and 17.2 on 32-row tiles).
//
// The high and the low terms' products have accumulators of their own (one term: even and odd groups), added at the end: chains
// half as long as in the kernel on 32-row tiles.
#include "zr_internal.h"
#include "zr_math.h"
#include "zr_mfma_core.h"

namespace {

constexpr int kWaves = 8;
constexpr int ROWS = 8;   // hidden rows of a workgroup
constexpr int kRedLd = 36;  // LDS row of 32 partial sums, padded

struct LstmRows16 {
  const unsigned short* W;     // [nseg][4] matrices of [H/8][ldw][8]
  const float* bias;           // [4][H]
  const unsigned short *hi[3], *lo[3];  // segment inputs, [H/8][mb][8]
  const float* cprev;
  const int* mask01;
  float *h, *c;
  float* gates[4];             // all null or all non-null
  unsigned short *out_hi, *out_lo;  // optional: h as bf16 terms, [H/8][mb][8]
  int nseg, H, mb, ldw, j_tiles, n_tiles;
  float clip;
};

// NARROW: 16 columns on the 16 x 16 x 32 instruction; else TN tiles of 32 columns on the 32 x 32 x 16 one.
// PF: k-groups in flight.
template <int TN, bool NARROW, bool LO, int PF>
__global__ void __launch_bounds__(64 * kWaves, 2) lstm_rows_bf16_kernel(LstmRows16 P) {
  static_assert(!NARROW || TN == 1, "tile shape");
  constexpr int KB = NARROW ? 4 : 2;            // k-blocks of 8 per k-group
  constexpr int NB = NARROW ? 2 : 1;            // weight sub-tiles
  constexpr int COLS = NARROW ? 16 : 32 * TN;
  constexpr int NOUT = (ROWS * COLS + 511) / 512;
  constexpr int NS = PF + 1;
  __shared__ float red[kWaves * COLS * kRedLd];
  // Workgroup ids congruent mod 8 share a die: the column tiles of a row tile, which read the same weights, go together.
  const int id = blockIdx.x;
  const int jt = (id / (8 * P.n_tiles)) * 8 + (id & 7);
  const int nt = (id >> 3) % P.n_tiles;
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
  float bias[NOUT][4], cprev_v[NOUT], mask_v[NOUT];
#pragma unroll
  for (int u = 0; u < NOUT; ++u) {
    const int o = tid + 512 * u;
    oj[u] = o % ROWS;
    on[u] = o / ROWS;
    const int j = j0 + oj[u], n = n0 + on[u];  // (H is a multiple of ROWS)
    ok[u] = o < ROWS * COLS && n < mb;
    const int nc = n < mb ? n : mb - 1;
#pragma unroll
    for (int g = 0; g < 4; ++g) bias[u][g] = P.bias[g * H + j];
    cprev_v[u] = P.cprev[(long long)nc * H + j];
    mask_v[u] = (float)P.mask01[nc];
  }

  unsigned xoff[TN], woff[NB];  // elements
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
    const int c = n0 + tn * 32 + cl;
    xoff[tn] = 8u * (unsigned)(c < mb ? c : mb - 1);
  }
  const unsigned HH = (unsigned)H * (unsigned)P.ldw;  // one matrix
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int c = cl + 16 * b;
    woff[b] = (unsigned)(c / ROWS) * HH + 8u * (unsigned)(j0 + c % ROWS);
  }
  const int kbs = H >> 3;                 // k-blocks of a segment
  const int G = (kbs + KB - 1) / KB;      // k-groups of a segment; the last narrow one may be half
  const int total = P.nseg * G;

  struct Frag {
    zr_u32x4 w[NB], hi[TN], lo[LO ? TN : 1];
    bool whole;
  };
  Frag f[NS];
  // The k-groups of all segments in one row, dealt to the waves in turn: group r is (segment r / G, group r % G).
  int ls = kslice / G, lg = kslice - ls * G, lr = kslice;  // the next group to load
  auto load = [&](Frag& q) {
    const unsigned short* Ws = P.W + 4ull * HH * (unsigned)ls;
    const int kb = KB * lg + kq;
    q.whole = !NARROW || kb < kbs;
    const unsigned kbc = (unsigned)(q.whole ? kb : kbs - 1);
#pragma unroll
    for (int b = 0; b < NB; ++b) q.w[b] = *(const zr_u32x4*)(Ws + (woff[b] + kbc * 8u * (unsigned)P.ldw));
    const unsigned xk = kbc * 8u * (unsigned)mb;
    const unsigned short *xh = P.hi[ls], *xl = P.lo[ls];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      q.hi[tn] = *(const zr_u32x4*)(xh + (xoff[tn] + xk));
      if constexpr (LO) q.lo[tn] = *(const zr_u32x4*)(xl + (xoff[tn] + xk));
    }
    // past the end: the last group again (not multiplied)
    if (lr + kWaves < total) {
      lr += kWaves;
      lg += kWaves;
      while (lg >= G) lg -= G, ++ls;
    }
  };
  zr_f32x16 acc[2][TN];
  zr_f32x4 acc4[2][NB];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[q][tn][r] = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b) acc4[q][b] = {0.0f, 0.0f, 0.0f, 0.0f};
  }
  auto mma = [&](Frag& q, int parity) {
    if (NARROW && !q.whole) {  // (both operands: zero times an infinite value is not zero)
      const zr_u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int b = 0; b < NB; ++b) q.w[b] = z;
      q.hi[0] = z;
      if constexpr (LO) q.lo[0] = z;
    }
#pragma unroll
    for (int p = 0; p < (LO ? 2 : 1); ++p) {
      const int a = LO ? p : parity & 1;
      if constexpr (NARROW) {
        const zr_bf16x8 x = __builtin_bit_cast(zr_bf16x8, LO && p == 1 ? q.lo[0] : q.hi[0]);
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc4[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(zr_bf16x8, q.w[b]), acc4[a][b], 0, 0, 0);
      } else {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const zr_bf16x8 x = __builtin_bit_cast(zr_bf16x8, LO && p == 1 ? q.lo[LO ? tn : 0] : q.hi[tn]);
          acc[a][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, __builtin_bit_cast(zr_bf16x8, q.w[0]), acc[a][tn], 0, 0, 0);
        }
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
        mma(f[s], s);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < PF; ++s)
      if (it + s < n_mine) mma(f[s], s);
  }

  // partial sums of the K slices through LDS, then the cell
  float* mine = red + kslice * (COLS * kRedLd);
  if constexpr (NARROW) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) mine[(4 * kq + r) * kRedLd + cl + 16 * b] = acc4[0][b][r] + acc4[1][b][r];
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
    zr_lstm_cell(z[0] + bias[u][0], z[1] + bias[u][1], z[2] + bias[u][2], z[3] + bias[u][3], cprev_v[u], mask_v[u], P.clip, gi, gf, gc, go, c, h);
    const int j = j0 + oj[u], n = n0 + on[u];
    const long long ix = (long long)n * H + j;
    P.c[ix] = c;
    P.h[ix] = h;
    if (P.out_hi) {
      const long long o = ((long long)(j >> 3) * mb + n) * 8 + (j & 7);
      const __bf16 hb = (__bf16)h;
      P.out_hi[o] = __builtin_bit_cast(unsigned short, hb);
      if (P.out_lo) P.out_lo[o] = __builtin_bit_cast(unsigned short, (__bf16)(h - (float)hb));
    }
    if (P.gates[0]) P.gates[0][ix] = gi, P.gates[1][ix] = gf, P.gates[2][ix] = gc, P.gates[3][ix] = go;
  }
}

template <bool LO>
void launch(const LstmRows16& P, int shape, unsigned grid, hipStream_t st) {
  switch (shape) {
    case 1: lstm_rows_bf16_kernel<1, true, LO, 8><<<grid, 64 * kWaves, 0, st>>>(P); break;
    case 2: lstm_rows_bf16_kernel<1, false, LO, 8><<<grid, 64 * kWaves, 0, st>>>(P); break;
    default: lstm_rows_bf16_kernel<2, false, LO, 6><<<grid, 64 * kWaves, 0, st>>>(P); break;
  }
}

}  // namespace

int zr_lstm_rows_bf16_step(zr_ctx* ctx, const zr_lstm_weights* w, int nseg, const unsigned short* const hi[3], const unsigned short* const lo[3],
                           const float* d_cprev, const int* d_mask01, float clip, int mb, float* d_h, float* d_c, float* const d_gates[4],
                           unsigned short* out_hi, unsigned short* out_lo, int shape) {
  LstmRows16 P = {};
  P.W = (const unsigned short*)w->d_W;
  P.bias = w->d_bias;
  for (int s = 0; s < nseg; ++s) P.hi[s] = hi[s], P.lo[s] = lo[s];
  P.cprev = d_cprev;
  P.mask01 = d_mask01;
  P.h = d_h;
  P.c = d_c;
  for (int g = 0; g < 4; ++g) P.gates[g] = d_gates ? d_gates[g] : nullptr;
  P.out_hi = out_hi;
  P.out_lo = out_lo;
  P.nseg = nseg;
  P.H = w->H;
  P.mb = mb;
  P.ldw = w->ldw;
  P.clip = clip;
  const int cols = shape == 1 ? 16 : (shape == 2 ? 32 : 64);
  P.j_tiles = P.H / ROWS;
  P.n_tiles = (mb + cols - 1) / cols;
  const unsigned grid = (unsigned)((P.j_tiles + 7) / 8 * 8 * P.n_tiles);
  if (lo[0])
    launch<true>(P, shape, grid, ctx->stream);
  else
    launch<false>(P, shape, grid, ctx->stream);
  ZR_LAUNCH_CHECK("lstm_rows_bf16_kernel");
  return ZR_OK;
}
