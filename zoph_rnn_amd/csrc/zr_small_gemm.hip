// Small products -- a few hundred to two thousand rows by a minibatch of columns, K up to a few thousand -- as narrow tiles
// whose operands are all on their way at once.
//
// The attention projections and output product, the error products of a node and of a diagonal of the backward sweep: 0.03 to
// 1 GFLOP over matrices that lie in the caches.  What bounds them is the launch, one trip to memory, and the chain of matrix
// instructions of a wave.  gemm_kernel's 32 x 32 tiles leave most of the chip idle (500 x 64 outputs: 32 workgroups), fetch a row-major or
// column-major matrix 4 bytes a lane and three groups of 8 k ahead, so that a wave makes several trips one after the other.
// Here a workgroup has 16 * TM x 16 * TN outputs, its eight waves take the groups of 16 k (32 with bf16 weights) of all segments in
// turn, and a wave has PF groups in flight, which for most of these products is all it has; the waves' sums are added
// through LDS in a fixed order.  Two accumulators an output (even and odd k) where a wave has one tile, so that an instruction need
// not wait for the one before; a sum is rounded in chains of K / 64 instructions.
#include "zr_internal.h"
#include "zr_mfma_core.h"

namespace {

constexpr int kWaves = 8;

struct SmallArgs {
  int M, N, K, nseg, epi, accum, batch, b_pack4;
  int m_tiles, n_tiles, rows;  // rows: row tiles of all problems
  const float* A[4];
  const float* B[4];
  const unsigned short* Blo[4];
  long long lda[4];
  int ldb[4];
  float* C;
  long long ldc, strideA, strideC, strideBias;
  const float* bias;
  const int* mask;
  float* Cpack;
  unsigned short *Chi, *Clo;
  int groups;
  const float* gA[8];
  const float* gB[8];
  float* gC[8];
  long long gStrideC[8];
};

typedef zr_f32x4 zr_f32x4_u __attribute__((aligned(4)));

// A column's four values from k0 on were read at `at` <= k0, the last place a whole load ends inside the column: shift them
// back, zeros behind the end.
__device__ __forceinline__ zr_f32x4 shifted(zr_f32x4 v, int d) {
  zr_f32x4 r;
  r[0] = d == 0 ? v[0] : (d == 1 ? v[1] : (d == 2 ? v[2] : (d == 3 ? v[3] : 0.0f)));
  r[1] = d == 0 ? v[1] : (d == 1 ? v[2] : (d == 2 ? v[3] : 0.0f));
  r[2] = d == 0 ? v[2] : (d == 1 ? v[3] : 0.0f);
  r[3] = d == 0 ? v[3] : 0.0f;
  return r;
}

// ONE: one segment, ungrouped.  No load then needs an entry of a table of arguments by a computed index, which took a second trip for arguments
// ahead of the first loads and others inside the loop: 885 x 126 x 98 5.0 -> 4.5 us, 1026 x 105 x 1030 11.7 -> 9.8, 2535 x 34 x 1463
// 15.7 -> 13.2.  Not for bf16 matrices: the compiler then keeps so many addresses in registers that some forms spill (a decode step at H = 1024, 64
// columns 122 -> 129 us).
template <int TM, int TN, int AMODE, int PF, bool ONE>
__global__ void __launch_bounds__(64 * kWaves, 2) small_gemm_kernel(SmallArgs a) {
  constexpr bool BF16 = zr_is_bf16_mode(AMODE), LO = AMODE == ZR_A_PACK8_BF16;
  constexpr int KG = BF16 ? 32 : 16;        // k of a group
  constexpr int NACC = TM * TN == 1 ? 2 : 1;
  constexpr int NOUT = TM * TN * 256 / 512 > 0 ? TM * TN * 256 / 512 : 1;
  constexpr int NS = PF + 1;
  __shared__ float red[kWaves][TM * TN * 4][64];
  // Workgroup ids congruent modulo 8 share a die: each die takes a contiguous range of the tiles, all column tiles of a row in turn.
  const int tiles = a.rows * a.n_tiles, per_die = (tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if (tile >= tiles) return;
  const int row_tile = tile / a.n_tiles, nt = tile - row_tile * a.n_tiles;
  const int z = row_tile / a.m_tiles, mt = row_tile - z * a.m_tiles;
  const int group = ONE ? 0 : z / a.batch, zb = z - group * a.batch;
  const int tid = threadIdx.x, lane = tid & 63, cl = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = 16 * TM * mt, n0 = 16 * TN * nt;
  float* C = !ONE && a.groups ? a.gC[group] + zb * a.gStrideC[group] : a.C + zb * a.strideC;
  const float* bias = a.bias ? a.bias + zb * a.strideBias : nullptr;

  // the outputs this thread finishes: what is added to them is fetched ahead of the K loop
  int om[NOUT], on[NOUT];
  bool ok[NOUT];
  float old[NOUT], add[NOUT], mask[NOUT];
#pragma unroll
  for (int u = 0; u < NOUT; ++u) {
    const int o = tid + 512 * u, s = o >> 6;  // s: tile * 4 + register
    om[u] = m0 + 16 * ((s >> 2) / TN) + cl;
    on[u] = n0 + 16 * ((s >> 2) % TN) + 4 * kq + (s & 3);
    ok[u] = o < TM * TN * 256 && om[u] < a.M && on[u] < a.N;
    old[u] = ok[u] && a.accum ? C[om[u] + on[u] * a.ldc] : 0.0f;
    add[u] = ok[u] && bias ? bias[om[u]] : 0.0f;
    mask[u] = ok[u] && a.epi == ZR_EPI_TANH_BIAS_MASK ? (float)a.mask[on[u]] : 0.0f;
  }

  int row[TM], col[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) row[i] = m0 + 16 * i + cl < a.M ? m0 + 16 * i + cl : a.M - 1;
#pragma unroll
  for (int j = 0; j < TN; ++j) col[j] = n0 + 16 * j + cl < a.N ? n0 + 16 * j + cl : a.N - 1;

  const int K = a.K, G = (K + KG - 1) / KG, total = ONE ? G : a.nseg * G;
  struct Frag {
    zr_f32x4 w[TM], x[TN], xl[LO ? TN : 1];
  };
  Frag f[NS];
  // The k-groups of all segments in one row, dealt to the waves in turn: group r is (segment r / G, group r % G).
  int ls = ONE ? 0 : wave / G, lg = wave - ls * G, lr = wave;  // the next group to load
  auto load = [&](Frag& q) {
    const float* A = !ONE && a.groups ? a.gA[group] : a.A[ls];
    const float* B = !ONE && a.groups ? a.gB[group] : a.B[ls];
    const long long lda = a.lda[ls], ldb = a.ldb[ls];
    if constexpr (BF16) {
      const int kb = 4 * lg + kq, last = (K >> 3) - 1, k8 = kb < last ? kb : last;
      const unsigned short* W = (const unsigned short*)A + zb * a.strideA;
#pragma unroll
      for (int i = 0; i < TM; ++i) q.w[i] = *(const zr_f32x4*)(W + (k8 * lda + row[i]) * 8);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const long long at = ((long long)k8 * a.N + col[j]) * 8;
        q.x[j] = *(const zr_f32x4*)((const unsigned short*)B + at);
        if (LO) q.xl[j] = *(const zr_f32x4*)(a.Blo[ls] + at);
      }
    } else {
      const float* W = A + zb * a.strideA;
      const int k0 = 16 * lg + 4 * kq, ks = k0 < K - 4 ? k0 : K - 4;
      if constexpr (AMODE == ZR_A_PACK4) {
        const int last = (K - 1) >> 2, kb = (k0 >> 2) < last ? (k0 >> 2) : last;
#pragma unroll
        for (int i = 0; i < TM; ++i) q.w[i] = *(const zr_f32x4*)(W + (kb * lda + row[i]) * 4);
        if (a.b_pack4) {
#pragma unroll
          for (int j = 0; j < TN; ++j) q.x[j] = *(const zr_f32x4*)(B + ((long long)kb * a.N + col[j]) * 4);
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) q.x[j] = *(const zr_f32x4_u*)(B + col[j] * ldb + ks);
        }
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if (AMODE == ZR_A_TRANS) {
            q.w[i] = *(const zr_f32x4_u*)(W + row[i] * lda + ks);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) q.w[i][e] = W[row[i] + (ks + e) * lda];
          }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) q.x[j] = *(const zr_f32x4_u*)(B + col[j] * ldb + ks);
      }
    }
    // past the end: the last group again (not multiplied)
    if (lr + kWaves < total) {
      lr += kWaves;
      lg += kWaves;
      if (!ONE)
        while (lg >= G) lg -= G, ++ls;
    }
  };

  zr_f32x4 acc[NACC][TM][TN] = {};
  int mg = ONE ? wave : wave % G;  // the group (inside its segment) multiplied next
  auto mma = [&](Frag& q) {
    if (KG * (mg + 1) > K) {  // K ends inside this group: shift the moved loads back, zeros behind the end in both operands
      if constexpr (BF16) {
        if (4 * mg + kq > (K >> 3) - 1) {
#pragma unroll
          for (int i = 0; i < TM; ++i) q.w[i] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            q.x[j] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (LO) q.xl[j] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
        }
      } else {
        const int k0 = 16 * mg + 4 * kq, d = k0 < K - 4 ? 0 : k0 - (K - 4);
        const int dp = k0 < K ? 0 : 4;  // k-interleaved operands: a whole block of 4 or none (rows past K hold zeros)
#pragma unroll
        for (int i = 0; i < TM; ++i) q.w[i] = shifted(q.w[i], AMODE == ZR_A_PACK4 ? dp : d);
#pragma unroll
        for (int j = 0; j < TN; ++j) q.x[j] = shifted(q.x[j], AMODE == ZR_A_PACK4 && a.b_pack4 ? dp : d);
      }
    }
    mg += kWaves;
    if (!ONE)
      while (mg >= G) mg -= G;
    if constexpr (BF16) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const zr_bf16x8 w = __builtin_bit_cast(zr_bf16x8, q.w[i]);
          acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(zr_bf16x8, q.x[j]), w, acc[0][i][j], 0, 0, 0);
          if (LO) {
            zr_f32x4& c = acc[NACC - 1][i][j];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(zr_bf16x8, q.xl[j]), w, c, 0, 0, 0);
          }
        }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            zr_f32x4& c = acc[e & (NACC - 1)][i][j];
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(q.x[j][e], q.w[i][e], c, 0, 0, 0);
          }
    }
  };
  if (wave < total) {
    const int n_mine = (total - wave + kWaves - 1) / kWaves;
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

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[0][i][j][r];
        if (NACC == 2) v += acc[NACC - 1][i][j][r];
        red[wave][(i * TN + j) * 4 + r][lane] = v;
      }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NOUT; ++u) {
    if (!ok[u]) continue;
    float p[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) p[w] = red[w][(tid + 512 * u) >> 6][lane];
    float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    const int m = om[u], n = on[u];
    float* c = C + m + n * a.ldc;
    if (a.epi == ZR_EPI_STORE) {
      v += add[u];
      *c = a.accum ? old[u] + v : v;
    } else if (a.epi == ZR_EPI_TANH) {
      *c = tanhf(v);
    } else {  // ZR_EPI_TANH_BIAS_MASK
      v = tanhf(v + add[u]) * mask[u];
      *c = v;
      if (a.Cpack) a.Cpack[((long long)(m >> 2) * a.N + n) * 4 + (m & 3)] = v;
      if (a.Chi) {  // the split of zr_split_bf16_pair, element by element
        const __bf16 hb = (__bf16)v;
        const long long o = ((long long)(m >> 3) * a.N + n) * 8 + (m & 7);
        a.Chi[o] = __builtin_bit_cast(unsigned short, hb);
        if (a.Clo) a.Clo[o] = __builtin_bit_cast(unsigned short, (__bf16)(v - (float)hb));
      }
    }
  }
}

template <int TM, int TN, int AMODE, int PF>
void launch_mode(const SmallArgs& a, unsigned grid, hipStream_t stream) {
  if constexpr (!zr_is_bf16_mode(AMODE)) {
    if (a.nseg == 1 && !a.groups) {
      small_gemm_kernel<TM, TN, AMODE, PF, true><<<grid, 64 * kWaves, 0, stream>>>(a);
      return;
    }
  }
  small_gemm_kernel<TM, TN, AMODE, PF, false><<<grid, 64 * kWaves, 0, stream>>>(a);
}

template <int TM, int TN, int PF>
void launch(const SmallArgs& a, int amode, unsigned grid, hipStream_t stream) {
  switch (amode) {
    case ZR_A_NN: launch_mode<TM, TN, ZR_A_NN, PF>(a, grid, stream); break;
    case ZR_A_TRANS: launch_mode<TM, TN, ZR_A_TRANS, PF>(a, grid, stream); break;
    case ZR_A_PACK4: launch_mode<TM, TN, ZR_A_PACK4, PF>(a, grid, stream); break;
    case ZR_A_PACK8_BF16: launch_mode<TM, TN, ZR_A_PACK8_BF16, PF>(a, grid, stream); break;
    default: launch_mode<TM, TN, ZR_A_PACK8_BF16_1T, PF>(a, grid, stream); break;
  }
}

}  // namespace

int zr_small_gemm(zr_ctx* ctx, const ZrGemmDesc& d, const unsigned short* const Bhi[4], const unsigned short* const Blo[4], int shape) {
  SmallArgs a = {};
  a.M = d.M, a.N = d.N, a.K = d.K[0], a.nseg = d.nseg;
  a.epi = d.epilogue, a.accum = d.accumulate, a.batch = d.batch, a.b_pack4 = d.b_packed;
  for (int s = 0; s < d.nseg; ++s) {
    a.A[s] = d.A[s], a.lda[s] = d.lda[s];
    a.B[s] = d.a_pack == 2 ? (const float*)Bhi[s] : d.B[s], a.ldb[s] = d.ldb[s];
    a.Blo[s] = d.a_pack == 2 ? Blo[s] : nullptr;
  }
  a.C = d.C, a.ldc = d.ldc;
  a.strideA = d.strideA, a.strideC = d.strideC, a.strideBias = d.strideBias;
  a.bias = d.bias, a.mask = d.mask, a.Cpack = d.Cpack, a.Chi = d.Chi, a.Clo = d.Clo;
  a.groups = d.groups;
  for (int g = 0; g < d.groups; ++g) a.gA[g] = d.gA[g], a.gB[g] = d.gB[g], a.gC[g] = d.gC[g], a.gStrideC[g] = d.gStrideC[g] ? d.gStrideC[g] : d.strideC;
  const int tm = shape == 2 ? 32 : 16, tn = shape == 0 ? 16 : 32;
  a.m_tiles = (d.M + tm - 1) / tm;
  a.n_tiles = (d.N + tn - 1) / tn;
  a.rows = a.m_tiles * d.batch * (d.groups > 0 ? d.groups : 1);
  const unsigned grid = (unsigned)(a.rows * a.n_tiles + 7) / 8 * 8;
  const int amode = d.a_pack == 2 ? (a.Blo[0] ? ZR_A_PACK8_BF16 : ZR_A_PACK8_BF16_1T)
                                  : (d.a_pack ? ZR_A_PACK4 : (d.trans_a ? ZR_A_TRANS : ZR_A_NN));
  switch (10 * shape + zr_small_gemm_depth(shape, a.K, a.nseg, d.a_pack)) {
    case 2: launch<1, 1, 2>(a, amode, grid, ctx->stream); break;
    case 4: launch<1, 1, 4>(a, amode, grid, ctx->stream); break;
    case 8: launch<1, 1, 8>(a, amode, grid, ctx->stream); break;
    case 13: launch<1, 2, 3>(a, amode, grid, ctx->stream); break;
    case 16: launch<1, 2, 6>(a, amode, grid, ctx->stream); break;
    default: launch<2, 2, 4>(a, amode, grid, ctx->stream); break;
  }
  ZR_LAUNCH_CHECK("small_gemm_kernel");
  return ZR_OK;
}
