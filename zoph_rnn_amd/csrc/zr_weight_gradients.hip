// Weight and bias gradients of one LSTM layer over all columns of its steps, for small models: dM = dg x^T, dWh = dg [h0, h_1 ..]^T and db = the sums
// of dg's rows, 4H x N times N x H with N = steps * minibatch, in one launch.
//
// Both operands have their rows contiguous for every column, which is how the matrix instruction wants them, so they are read as they lie: the older
// route transposed the right-hand sides into scratch memory, multiplied twice and summed the rows, seven launches.  A workgroup has
// 64 x 64 outputs; its eight waves take the columns in turn, sixteen at a time, two 32 x 32 tiles either way each, and the waves' sums are added
// through LDS in a fixed order.  Two accumulators an output, for every other instruction: a sum is rounded in chains of N / 32
// instructions (with one its error against 64 bits was up to 30 % above the older route's).
// Bound: the matrix cores in fp32 where the tiles fill the chip, else the operands' way from L2.  2 x (1200 x 300 x 700) 40 -> 21 us, 2 x (2000 x 500 x 1536) 99 -> 78 (the older
// route on the bf16 matrix cores), 2 x (1200 x 300 x 64) 18 -> 6.5.
#include "zr_internal.h"

namespace {

constexpr int kWaves = 8;
constexpr int kStep = 16;  // columns a wave takes at a time

struct WeightGrads {
  const float* dg;     // [N][4H]
  const float* in;     // [N][H]
  const float* h0;     // [mb][H]: the first mb columns of the other right-hand side ...
  const float* h_all;  // ... and the rest
  float *dM, *dWh, *db;
  int H, mb, N, accumulate, m_tiles, n_tiles;
};

__global__ void __launch_bounds__(64 * kWaves, 2) weight_gradients_kernel(WeightGrads P) {
  __shared__ float red[kWaves][16][64];
  const int H = P.H, M = 4 * H, N = P.N;
  // Workgroup ids congruent modulo 8 share a die: each takes a contiguous range of the tiles, all of a row of dg in turn.
  const int tiles = P.m_tiles * P.n_tiles * 2, per_die = (tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int mt = tile / (2 * P.n_tiles), rest = tile - mt * 2 * P.n_tiles, z = rest / P.n_tiles, nt = rest - z * P.n_tiles;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = 64 * mt, n0 = 64 * nt;
  unsigned am[2], bn[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    am[i] = (unsigned)(m0 + 32 * i + r < M ? m0 + 32 * i + r : M - 1);
    bn[i] = (unsigned)(n0 + 32 * i + r < H ? n0 + 32 * i + r : H - 1);
  }
  const bool bias = z == 0 && nt == 0;
  constexpr int U = kStep / 2;
  float av[U][2], bv[U][2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 2 * u + half;
      const bool in = k < N;
      const int kk = in ? k : N - 1;
      const float* a = P.dg + (size_t)kk * M;
      const float* b = z == 0 ? P.in + (size_t)kk * H : (kk < P.mb ? P.h0 + (size_t)kk * H : P.h_all + (size_t)(kk - P.mb) * H);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float x = a[am[i]], y = b[bn[i]];
        av[u][i] = in ? x : 0.0f;
        bv[u][i] = in ? y : 0.0f;
      }
    }
  };
  zr_f32x16 acc[2][2][2] = {};
  float rows[2] = {0.0f, 0.0f};
  int k0 = kStep * wave;
  if (k0 < N) fetch(k0);
  for (; k0 < N; k0 += kStep * kWaves) {
    float ac[U][2], bc[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) ac[u][i] = av[u][i], bc[u][i] = bv[u][i];
    if (k0 + kStep * kWaves < N) fetch(k0 + kStep * kWaves);
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[u & 1][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bc[u][j], ac[u][i], acc[u & 1][i][j], 0, 0, 0);
    }
    if (bias)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        rows[i] += ((ac[0][i] + ac[1][i]) + (ac[2][i] + ac[3][i])) + ((ac[4][i] + ac[5][i]) + (ac[6][i] + ac[7][i]));
  }

  float* C = z == 0 ? P.dM : P.dWh;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 16; ++q) red[wave][q][lane] = acc[0][i][j][q] + acc[1][i][j][q];
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int q = (tid >> 6) + 8 * u;
        const int m = m0 + 32 * i + r, n = n0 + 32 * j + 8 * (q >> 2) + 4 * half + (q & 3);
        if (m >= M || n >= H) continue;
        float part[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) part[w] = red[w][q][lane];
        const float sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        float* c = C + (size_t)n * M + m;
        *c = P.accumulate ? *c + sum : sum;
      }
    }
  if (!bias) return;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) red[wave][i][lane] = rows[i];
  __syncthreads();
  if (tid >= 64 || m0 + tid >= M) return;
  float sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum += red[w][tid >> 5][r] + red[w][tid >> 5][32 + r];
  P.db[m0 + tid] = P.accumulate ? P.db[m0 + tid] + sum : sum;
}

}  // namespace

int zr_weight_gradients(zr_ctx* ctx, int H, int N, int mb, const float* d_dgates, const float* d_in_all, const float* d_h0, const float* d_h_all,
                        float* d_dM, float* d_dWh, float* d_db, int accumulate) {
  WeightGrads P = {d_dgates, d_in_all, d_h0, d_h_all, d_dM, d_dWh, d_db, H, mb, N, accumulate, (4 * H + 63) / 64, (H + 63) / 64};
  const unsigned grid = (unsigned)(((long long)P.m_tiles * P.n_tiles * 2 + 7) / 8 * 8);
  weight_gradients_kernel<<<grid, 64 * kWaves, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("weight_gradients_kernel");
  return ZR_OK;
}
