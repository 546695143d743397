// The output layer's product on a prepared fp32 matrix, V x H times H x columns, beyond 16 columns: the bf16 matrix cores with every operand as
// three exact bf16 terms (zr_split_gemm.hip says why that loses nothing), the matrix straight from memory into the registers
// of the one wave that multiplies it.
//
// A wave owns 32 rows and all 32 * TN columns of its workgroup's tile: its fragments of the matrix are two 16-byte loads a lane for 16 k in
// the k-interleaved layout, PD steps of 32 k ahead, split into terms in registers and never shared, so every element of the
// matrix is fetched and converted once per column tile.  The activations' 32 k are read as they lie, split by all threads on their way
// into LDS, one step ahead, and read by all waves.  The twelve products of 32 k are added up from zero and their sum is added to the
// accumulator: short chains, one rounding at the accumulator's size.  An accumulator that comes out infinite or NaN is computed again with
// fp32 instructions (the terms of an infinite operand are infinity and NaN).
// Bound by matrix instructions and conversions together: at 50000 x 128 x 1000 the matrix pipes of the 200 compute units that have a tile are busy for 57 %,
// the vector instructions take 44 % of their cycles.  It takes 89 to 92 us (12.8 GFLOP, 77 of bf16 work); the fp32 instructions took 110 to
// 124; 64 columns of 30011 x 500 31 -> 22, 32 columns 20.9 -> 17.2, of 50000 x 300 27.3 -> 15.9.
// Error of the logits against 64 bits, relative 2-norm, here and with the fp32 instructions: H = 64 7.6e-8 / 8.7e-8, 200 9.1e-8 / 1.36e-7, 500
// 1.09e-7 / 2.06e-7, 1000 1.35e-7 / 2.1e-7 to 2.9e-7.
// Tried and dropped at 128 columns: one chain of dependent instructions a column block instead of two in turn (107 against 103 us the whole
// call), the matrix split a step ahead (spills), activations two steps ahead (106), two groups of waves in opposite phases, one
// splitting while the other multiplies (108).
#include "zr_internal.h"
#include "zr_logits_epilogue.h"
#include "zr_mfma_core.h"

namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any multiple of 4

struct LogitsArgs {
  int M, N, K, ldp, kp;  // A: element (row, k) at ((k/4)*ldp + row)*4 + k%4, k < kp
  const float* A;
  const float* B;        // column n at n*ldb
  long long ldb;
  float* C;
  long long ldc;
  const float* bias;
  float* partials;
  int m_tiles, n_tiles;
};

constexpr int KC = 32;  // k of a step

// Where column c of a k-group lies: the four k-groups are turned against each other, so that neither a fragment's read (two
// k-groups at a time) nor a store (all four) finds two of its items in the same banks.
__device__ __forceinline__ int turned(int c, int kg) { return c ^ (8 * (kg & 1) + 4 * (kg >> 1)); }

template <int TN, int W, int PD, int WAUX>
__global__ void __launch_bounds__(64 * W, 2) logits_split_kernel(LogitsArgs a) {
  constexpr int COLS = 32 * TN, KG = COLS, TERM = 4 * KG, BUF = 3 * TERM;
  constexpr int ITEMS = 4 * COLS, NI = (ITEMS + 64 * W - 1) / (64 * W);  // (k-group, column) pairs of a step, of a thread
  __shared__ zr_u32x4 s[2 * BUF];
  const int tid = threadIdx.x, lane = tid & 63, jl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup ids congruent modulo 8 share a die: each takes a contiguous range of the tiles, all column tiles of a row tile in turn.
  const int tiles = a.m_tiles * a.n_tiles, per_die = (tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int mt = tile / a.n_tiles;
  const int m0 = (mt * W + wave) * 32, n0 = (tile - mt * a.n_tiles) * COLS;
  const int row = m0 + jl < a.M ? m0 + jl : a.M - 1;
  const int steps = (a.K + KC - 1) / KC;

  // The matrix through a descriptor that ends with it: what lies past kp reads as zero.
  const __amdgpu_buffer_rsrc_t arsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.A), 0, (int)(unsigned)((long long)a.kp * a.ldp * 4), 0x00020000);
  const unsigned kstep = 16u * (unsigned)a.ldp;  // bytes of four k
  const unsigned aoff = 16u * (unsigned)row + 2u * (unsigned)half * kstep;
  zr_f32x4 ar[PD + 1][4];
  auto load_a = [&](zr_f32x4 (&v)[4], int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i)  // blocks of four k: 0, 1, 4, 5 (half 0), 2, 3, 6, 7 (half 1)
      v[i] = __builtin_bit_cast(zr_f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              arsrc, (int)(aoff + (unsigned)(8 * c + (i & 1) + 4 * (i >> 1)) * kstep), 0, WAUX));
  };
  zr_f32x4 bv[NI][2];
  auto load_b = [&](int c) {
    const int k0 = c * KC;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int item = tid + 64 * W * i, kg = item & 3;
      if (ITEMS % (64 * W) != 0 && item >= ITEMS) break;  // uniform over a wave
      const int col = n0 + (item >> 2) < a.N ? n0 + (item >> 2) : a.N - 1;
      const float* q = a.B + (long long)col * a.ldb;
      if (k0 + KC <= a.K) {  // uniform
        bv[i][0] = *(const f32x4u*)(q + k0 + 8 * kg);
        bv[i][1] = *(const f32x4u*)(q + k0 + 8 * kg + 4);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = k0 + 8 * kg + j;
          const float x = q[k < a.K ? k : a.K - 1];
          bv[i][j >> 2][j & 3] = k < a.K ? x : 0.0f;
        }
      }
    }
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int item = tid + 64 * W * i, kg = item & 3;
      if (ITEMS % (64 * W) != 0 && item >= ITEMS) break;
      zr_u32x4 term[3];
      zr_split_terms(bv[i][0], bv[i][1], term);
      zr_u32x4* d = s + buf * BUF + kg * KG + turned(item >> 2, kg);
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q * TERM] = term[q];
    }
  };

  zr_f32x16 acc[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
  auto compute = [&](const zr_f32x4 (&v)[4], int buf) {
    zr_bf16x8 x[2][3];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      zr_u32x4 term[3];
      zr_split_terms(v[2 * st], v[2 * st + 1], term);
#pragma unroll
      for (int q = 0; q < 3; ++q) x[st][q] = __builtin_bit_cast(zr_bf16x8, term[q]);
    }
    // Two column blocks' chains in turn: an instruction that reads the sum of the one before waits for it twice as long as it takes.
#pragma unroll
    for (int j = 0; j < TN; j += 2) {
      zr_f32x16 sum[2] = {};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        zr_bf16x8 y[2][3];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (j + t >= TN) break;
          const zr_u32x4* b = s + buf * BUF + (2 * st + half) * KG + turned(32 * (j + t) + jl, 2 * st + half);
#pragma unroll
          for (int q = 0; q < 3; ++q) y[t][q] = __builtin_bit_cast(zr_bf16x8, b[q * TERM]);
        }
        constexpr int P[6] = {2, 0, 1, 1, 0, 0}, Q[6] = {0, 2, 1, 0, 1, 0};  // the smallest products first
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            if (j + t < TN) sum[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[st][P[p]], y[t][Q[p]], sum[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (j + t < TN) acc[j + t] += sum[t];
    }
  };

  load_b(0);
#pragma unroll
  for (int c = 0; c < PD; ++c) load_a(ar[c], c);
  store_b(0);
  if (steps > 1) load_b(1);
  __syncthreads();
  for (int c0 = 0; c0 < steps; c0 += PD + 1) {
#pragma unroll
    for (int u = 0; u < PD + 1; ++u) {
      const int c = c0 + u;
      if (c >= steps) break;  // uniform
      load_a(ar[(u + PD) % (PD + 1)], c + PD);
      // the other buffer was last read in step c - 1, behind the barrier that ended it
      if (c + 1 < steps) store_b((c + 1) & 1);
      if (c + 2 < steps) load_b(c + 2);
      compute(ar[u], c & 1);
      __syncthreads();
    }
  }

  if (m0 >= a.M) return;
  bool finite = true;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) finite = finite && fabsf(acc[j][r]) <= 3.402823466e38f;
  if (__any(!finite)) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    for (int k = 0; k < a.K; k += 2) {
      const bool in = k + half < a.K;
      const int kk = in ? k + half : k;
      const float xv = a.A[((long long)(kk >> 2) * a.ldp + row) * 4 + (kk & 3)], x = in ? xv : 0.0f;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + 32 * j + jl < a.N ? n0 + 32 * j + jl : a.N - 1;
        const float yv = a.B[n * a.ldb + kk];
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, in ? yv : 0.0f, acc[j], 0, 0, 0);
      }
    }
  }

  zr_logits_epilogue<TN>(acc, m0, n0, a.M, a.N, a.C, a.ldc, a.bias, a.partials, lane);
}

template <int TN, int W, int PD>
void launch(const LogitsArgs& a, bool stream, unsigned grid, hipStream_t st) {
  if (stream)
    logits_split_kernel<TN, W, PD, ZR_AUX_STREAM><<<grid, 64 * W, 0, st>>>(a);
  else
    logits_split_kernel<TN, W, PD, 0><<<grid, 64 * W, 0, st>>>(a);
}

template <int W>
void launch_tn(const LogitsArgs& a, int tn, bool stream, unsigned grid, hipStream_t st) {
  switch (tn) {
    case 1: launch<1, W, 3>(a, stream, grid, st); break;
    case 2: launch<2, W, 3>(a, stream, grid, st); break;
    case 3: launch<3, W, 2>(a, stream, grid, st); break;
    case 4: launch<4, W, 2>(a, stream, grid, st); break;
    case 5: launch<5, W, 1>(a, stream, grid, st); break;
    default: launch<6, W, 1>(a, stream, grid, st); break;
  }
}

}  // namespace

int zr_logits_split(zr_ctx* ctx, int V, int cols, int H, const float* packed, int ldp, const float* h, long long ldh, float* C,
                    long long ldc, const float* bias, float* partials, bool stream, int tn, int waves) {
  LogitsArgs a = {};
  a.M = V, a.N = cols, a.K = H, a.ldp = ldp, a.kp = (H + 7) / 8 * 8;
  a.A = packed, a.B = h, a.ldb = ldh, a.C = C, a.ldc = ldc, a.bias = bias, a.partials = partials;
  a.m_tiles = (V + 32 * waves - 1) / (32 * waves);
  a.n_tiles = (cols + 32 * tn - 1) / (32 * tn);
  const unsigned grid = (unsigned)(((long long)a.m_tiles * a.n_tiles + 7) / 8 * 8);
  if (waves == 8)
    launch_tn<8>(a, tn, stream, grid, ctx->stream);
  else
    launch_tn<4>(a, tn, stream, grid, ctx->stream);
  ZR_LAUNCH_CHECK("logits_split_kernel");
  return ZR_OK;
}
