// The error products of a diagonal of the backward sweep -- (error to h_{t-1}, error to the layer below) of up to eight nodes, each M x K times
// K x N with K = 4M -- on the bf16 matrix cores with every operand as three exact bf16 terms (zr_mma_segment_split).
//
// A workgroup has 64 x 64 outputs of one product, its four waves take the groups of 8 k in turn, straight from the k-interleaved copies of
// both operands into registers, and split what they multiply; their sums are added through LDS in a fixed order.  A die takes a contiguous
// range of the tiles, all column tiles of a row in turn, so that its level-two cache sees every element of the matrices once.
// Bound by the conversions beside the matrix instructions (61 % of a SIMD's cycles and 48.5 %, one wave a SIMD): a full diagonal of 4 layers of H = 1000 at 128
// columns (8.2 GFLOP) takes 81 us on the fp32 instructions and 53 to 57 here (the sweep of 12 steps 1190 -> 922).  Error of a product against 64 bits, here and
// there: H = 300 1.3e-7 to 1.6e-7 / 1.9e-7 to 2.4e-7, 1000 1.4e-7 to 2.6e-7 / 3.5e-7 to 4.7e-7 (with one chain of sums 3.7e-7).
#include "zr_internal.h"
#include "zr_mfma_core.h"

namespace {

struct ErrorProducts {
  const float* A[8];
  const float* B[8];
  float* C[8];
  long long strideA, strideC[8], ldc;
  int M, N, K, ldp, batch, products, m_tiles, n_tiles;
};

__global__ void __launch_bounds__(256, 1) error_products_kernel(ErrorProducts P) {
  constexpr int KS = 4, RING = 8;
  __shared__ float red[KS][4][16][64];
  const int tiles = P.products * P.m_tiles * P.n_tiles, per_die = (tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int nt = tile % P.n_tiles, row_tile = tile / P.n_tiles, z = row_tile / P.m_tiles, mt = row_tile - z * P.m_tiles;
  const int group = z / P.batch, zb = z - group * P.batch;
  const int lane = threadIdx.x & 63, jl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = 64 * mt, n0 = 64 * nt;
  const __amdgpu_buffer_rsrc_t wrsrc = zr_make_rsrc(P.A[group] + zb * P.strideA), xrsrc = zr_make_rsrc(P.B[group]);
  // rows past the copy's end (a multiple of 32): the first 32 again, not stored
  const unsigned wsoff[2] = {0u, m0 + 32 < P.ldp ? 512u : 0u};
  const unsigned woffb = 16u * (unsigned)(m0 + jl + half * P.ldp);
  unsigned xoffb[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int n = n0 + 32 * t + jl < P.N ? n0 + 32 * t + jl : P.N - 1;
    xoffb[t] = 16u * (unsigned)(n + half * P.N);
  }
  zr_f32x16 acc[2][2];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.0f;
  };
  clear();
  {
    ZrFrag<2, 2> ring[RING];
    zr_mma_segment_split<2, 2, KS, RING>(acc, wrsrc, wsoff, woffb, 32u * (unsigned)P.ldp, xrsrc, xoffb, 32u * (unsigned)P.N, P.K, wave, ring);
  }
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) finite = finite && fabsf(acc[i][t][r]) <= 3.402823466e38f;
  if (__any(!finite)) {
    clear();
    zr_mma_segment_ring<2, 2, KS, 2>(acc, wrsrc, wsoff, woffb, 32u * (unsigned)P.ldp, xrsrc, xoffb, 32u * (unsigned)P.N, P.K, wave);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave][2 * i + t][r][lane] = acc[i][t][r];
  __syncthreads();
  // wave w stores block w: a lane has one row and sixteen of the columns
  const int m = m0 + 32 * (wave >> 1) + jl;
  float* C = P.C[group] + zb * P.strideC[group];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int n = n0 + 32 * (wave & 1) + 8 * (r >> 2) + 4 * half + (r & 3);
    const float v = (red[0][wave][r][lane] + red[1][wave][r][lane]) + (red[2][wave][r][lane] + red[3][wave][r][lane]);
    if (m < P.M && n < P.N) C[m + n * P.ldc] = v;
  }
}

}  // namespace

int zr_error_products(zr_ctx* ctx, const ZrGemmDesc& d) {
  ErrorProducts P = {};
  for (int g = 0; g < d.groups; ++g)
    P.A[g] = d.gA[g], P.B[g] = d.gB[g], P.C[g] = d.gC[g], P.strideC[g] = d.gStrideC[g] ? d.gStrideC[g] : d.strideC;
  P.strideA = d.strideA, P.ldc = d.ldc;
  P.M = d.M, P.N = d.N, P.K = d.K[0], P.ldp = d.lda[0], P.batch = d.batch, P.products = d.groups * d.batch;
  P.m_tiles = (d.M + 63) / 64, P.n_tiles = (d.N + 63) / 64;
  const long long tiles = (long long)P.products * P.m_tiles * P.n_tiles;
  error_products_kernel<<<(unsigned)((tiles + 7) / 8 * 8), 256, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("error_products_kernel");
  return ZR_OK;
}
