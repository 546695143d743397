// Large fp32 products on the bf16 matrix cores, without giving up any of the operands' 24 bits.
//
// x = x1 + x2 + x3 with x1 = x rounded to bf16, x2 = x - x1 rounded to bf16 and x3 the rest, which has at most 8 bits:
// every subtraction is exact and nothing of x is lost while the third term is a normal number, |x| above about 2^-110.
// x*y is taken as the six products x1y1, x1y2, x2y1, x2y2, x1y3 and x3y1 (the three left out are below 2^-24 of x*y and of
// either sign), each exact, summed in the fp32 accumulator.  (A product below about 2^-100 has its smaller terms among the
// subnormal numbers: its absolute error is of that size.)  A sum of many terms carries no more error than with the fp32
// instructions; a sum that is one large term may carry three roundings of it instead of one.
// Six 32x32x16 bf16 instructions take 192 cycles of a matrix core for the work of eight 32x32x2 fp32 ones at 64 cycles
// each.  Against 64 bits, normal operands, relative 2-norm, beside the fp32 instructions': K = 500 3.3e-7 / 3.8e-7, 1000
// 4.7e-7 / 5.5e-7, 6400 1.3e-6 / 1.4e-6, 50000 1.9e-6 / 4.0e-6.
//
// What bounds it: the conversion (11 vector instructions for two values' three terms) and the LDS traffic beside the
// matrix cores, which are busy 51 to 66 % of the time in the products of a large training step and 26 to 54 % in smaller
// launches (a third of the cycles LDS is busy are bank conflicts).  The operands are read as fp32, as they lie, and split
// on their way into LDS, 32 k at a time; every fragment read from LDS then feeds several of the six products.  A workgroup
// of four waves has a tile of 128 x 128 (64 x 64 a wave, three workgroups a compute unit) or 128 x 256 (64 x 128 a wave,
// two), one LDS buffer, and the next step's values in registers while it multiplies: the workgroups of a compute unit cover
// each other's conversions and barriers.  50000 x 6400 x 1000: 128 x 128 tiles 3.94 ms, 128 x 256 3.49 (184 TFLOP/s of fp32 work;
// the fp32 instructions' kernel 5.70); 4000 x 1000 x 6400 0.47 -> 0.31; 33333 x 700 x 500 0.60 -> 0.16.
#include "zr_internal.h"
#include "zr_mfma_core.h"

namespace {

typedef zr_bf16x8 bf16x8;
typedef zr_u32x4 u32x4;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any multiple of 4

struct SplitArgs {
  int M, N, K;
  const float* A;
  const float* B;
  long long lda, ldb;
  float* C;
  long long ldc;
  const float* bias;
  float* partials;
  int accum;
  int m_tiles, n_tiles, parts, k_part;
  float* work;
};

constexpr int KC = 32;  // k values per step
constexpr int TM = 128; // rows of a workgroup's tile

// One operand in LDS: [term][k-group of 8][row], 16 bytes an item.
template <int ROWS>
struct Oper {
  static constexpr int KG = ROWS, TERM = 4 * KG, SIZE = 3 * TERM;
};

// Where row r of an operand's tile lies inside a k-group.  The low two bits are turned by (r / 16) % 4, so that threads
// that each store one row of four (rows 4q + j, one j at a time) hit different banks.  The k-groups are turned against each
// other by 8 and 4 items: a read of a fragment serves rows of two neighbouring k-groups at a time (one per half of the
// wave; with the groups 4 items apart half of every read met a conflict), a store threads of all four.
__device__ __forceinline__ int lds_row(int r, int kg) {
  return ((r & ~3) | ((r + (r >> 4)) & 3)) ^ (8 * (kg & 1) + 4 * (kg >> 1));
}

// One operand's share of a step, ROWS rows x 32 k, by 256 threads.
// ZR_SPLIT_K_FAST:   element (row, k) at p[row*ld + k]; a thread holds k-group t%4 of rows t/4 + 64*i, v[2*i + k%8/4][k%4].
// ZR_SPLIT_PACK4:    element (row, k) at p[(k/4*ld + row)*4 + k%4], k padded with zeros to a multiple of 8; a thread
//                    holds k-group t/64 of rows t%64 + 64*i, the same way.
// ZR_SPLIT_ROW_FAST: element (row, k) at p[row + k*ld]; a thread holds rows 4*(t/2%32) + 128*i + 0..3 at four k from
//                    4*(t%2 + 2*(t/64)), v[4*i + k%4][row%4].
template <int ROWS, int LAYOUT>
__device__ __forceinline__ void load_operand(f32x4u (&v)[ROWS / 32], const float* __restrict__ p, long long ld, int row0,
                                             int rows, int k0, int k_end, int t) {
  if (LAYOUT == ZR_SPLIT_PACK4) {
    const int k = k0 + 8 * (t >> 6);
    const bool in = k < k_end;
#pragma unroll
    for (int i = 0; i < ROWS / 64; ++i) {
      const int r = row0 + (t & 63) + 64 * i;
      const f32x4u* q = (const f32x4u*)p + (long long)(in ? k >> 2 : 0) * ld + (r < rows ? r : rows - 1);
      const f32x4u lo = q[0], hi = q[ld];
      v[2 * i] = in ? lo : f32x4u{0.0f, 0.0f, 0.0f, 0.0f};
      v[2 * i + 1] = in ? hi : f32x4u{0.0f, 0.0f, 0.0f, 0.0f};
    }
  } else if (LAYOUT == ZR_SPLIT_K_FAST) {
    if (k0 + KC <= k_end) {  // uniform
#pragma unroll
      for (int i = 0; i < ROWS / 64; ++i) {
        const int r = row0 + (t >> 2) + 64 * i;
        const float* q = p + (long long)(r < rows ? r : rows - 1) * ld + k0 + 8 * (t & 3);
        v[2 * i] = *(const f32x4u*)q;
        v[2 * i + 1] = *(const f32x4u*)(q + 4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < ROWS / 64; ++i) {
        const int r = row0 + (t >> 2) + 64 * i;
        const float* q = p + (long long)(r < rows ? r : rows - 1) * ld;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = k0 + 8 * (t & 3) + j;
          const float x = q[k < k_end ? k : k_end - 1];
          v[2 * i + j / 4][j & 3] = k < k_end ? x : 0.0f;
        }
      }
    }
  } else {
    const int kq = k0 + 4 * ((t & 1) + 2 * (t >> 6));
#pragma unroll
    for (int i = 0; i < ROWS / 128; ++i) {
      const int r = row0 + 4 * ((t >> 1) & 31) + 128 * i;
      if (k0 + KC <= k_end && row0 + 128 * i + 128 <= rows) {  // uniform
        const float* q = p + r + (long long)kq * ld;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * i + j] = *(const f32x4u*)(q + j * ld);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = kq + j;
          const float* q = p + (long long)(k < k_end ? k : k_end - 1) * ld;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = q[r + e < rows ? r + e : rows - 1];
            v[4 * i + j][e] = k < k_end ? x : 0.0f;
          }
        }
      }
    }
  }
}

template <int ROWS, int LAYOUT>
__device__ __forceinline__ void store_operand(u32x4* s, const f32x4u (&v)[ROWS / 32], int t) {
  typedef Oper<ROWS> O;
  if (LAYOUT != ZR_SPLIT_ROW_FAST) {
#pragma unroll
    for (int i = 0; i < ROWS / 64; ++i) {
      u32x4* d = LAYOUT == ZR_SPLIT_PACK4 ? s + (t >> 6) * O::KG + lds_row((t & 63) + 64 * i, t >> 6)
                                          : s + (t & 3) * O::KG + lds_row((t >> 2) + 64 * i, t & 3);
      u32x4 term[3];
      const zr_f32x4 lo = v[2 * i], hi = v[2 * i + 1];
      zr_split_terms(lo, hi, term);
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q * O::TERM] = term[q];
    }
  } else {
#pragma unroll
    for (int i = 0; i < ROWS / 128; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        u32x2* d = (u32x2*)(s + (t >> 6) * O::KG + lds_row(4 * ((t >> 1) & 31) + 128 * i + e, t >> 6)) + (t & 1);
        u32x2 term[3];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          float a = v[4 * i + 2 * p][e], b = v[4 * i + 2 * p + 1][e];
#pragma unroll
          for (int q = 0; q < 3; ++q) term[q][p] = zr_next_terms(a, b);
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) d[q * O::TERM * 2] = term[q];
      }
  }
}

template <int LAYOUT>
__device__ __forceinline__ long long element(long long row, long long k, long long ld) {
  return LAYOUT == ZR_SPLIT_PACK4 ? ((k >> 2) * ld + row) * 4 + (k & 3) : LAYOUT == ZR_SPLIT_K_FAST ? row * ld + k : row + k * ld;
}

// The same sums with fp32 instructions straight from memory: for a wave whose accumulators came out infinite or NaN.
// The terms of an infinite operand are infinity and NaN, so only this says what the sum of the operands' products is.
// It is the slow way, for the waves concerned only: 4000 x 1000 x 6400 takes 319 us, 748 with one NaN in A, 945 with one
// in B, 1049 with nothing finite in B (the fp32 kernels 500 in every case); 20000 x 6400 x 1000 1507, 1871, 1720, 4991 (2130).
template <int TNW, int AL, int BL, bool ROWS_FIRST>
__device__ __forceinline__ void plain_tile(const SplitArgs& a, zr_f32x16 (&acc)[2][TNW], int m0, int n0, int k_begin,
                                           int k_end, int lane) {
  const int jl = lane & 31, half = lane >> 5;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TNW; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  for (int k = k_begin; k < k_end; k += 2) {
    const bool in = k + half < k_end;
    const long long kk = in ? k + half : k;
    float x[2], y[TNW];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const long long m = m0 + 32 * i + jl < a.M ? m0 + 32 * i + jl : a.M - 1;
      const float xv = a.A[element<AL>(m, kk, a.lda)];
      x[i] = in ? xv : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < TNW; ++j) {
      const long long n = n0 + 32 * j + jl < a.N ? n0 + 32 * j + jl : a.N - 1;
      const float yv = a.B[element<BL>(n, kk, a.ldb)];
      y[j] = in ? yv : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < TNW; ++j)
        acc[i][j] = ROWS_FIRST ? __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], y[j], acc[i][j], 0, 0, 0)
                               : __builtin_amdgcn_mfma_f32_32x32x2f32(y[j], x[i], acc[i][j], 0, 0, 0);
  }
}

template <int TNW, int AL, int BL, int EPI>
__global__ void __launch_bounds__(256, TNW == 2 ? 3 : 2) split_gemm_kernel(SplitArgs a) {
  constexpr int TN = 64 * TNW;
  // The six products of 16 k are added up from zero and their sum is added to the accumulator: one rounding at its size where
  // the products one by one make six.  For the logits of a prepared output layer, whose fp32 kernel divides K over four waves.
  // Error of the probabilities against 64 bits at V = 50000, H = 1000, 257 to 1024 columns 4.3e-7 there, 1.0e-6 without
  // this, 3.4e-7 with it; H = 500 2.1e-7, 4.1e-7, 1.9e-7.  It costs up to 19 % (50000 x 1000, 400 columns 346 -> 413 us, 512 367 ->
  // 425; the fp32 kernel 473 there).  The other fp32 kernels' sums are no shorter than those of the products one by one.
  constexpr bool SHORT = AL == ZR_SPLIT_PACK4 && EPI == ZR_EPI_SOFTMAX_PARTIAL;
  typedef Oper<TM> OA;
  typedef Oper<TN> OB;
  __shared__ u32x4 s[OA::SIZE + OB::SIZE];
  const int tid = threadIdx.x, lane = tid & 63, jl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup ids congruent modulo 8 share an XCD: each takes a contiguous range of the tiles, which run through groups
  // of eight row tiles by all column tiles, so that the tiles in flight on an XCD share their operands in its L2.
  const int tiles = a.m_tiles * a.n_tiles;
  const int per_xcd = (tiles * a.parts + 7) >> 3;
  const int id = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || id >= tiles * a.parts) return;
  const int part = id / tiles, in_part = id - part * tiles;
  const int group = in_part / (8 * a.n_tiles), in_group = in_part - group * 8 * a.n_tiles;
  const int high = min(8, a.m_tiles - 8 * group);
  const int m0 = (8 * group + in_group % high) * TM, n0 = in_group / high * TN;
  const int k_begin = part * a.k_part, k_end = min(a.K, k_begin + a.k_part);

  zr_f32x16 acc[2][TNW];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TNW; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  f32x4u va[TM / 32], vb[TN / 32];
  const int wm = 64 * (wave & 1), wn = 32 * TNW * (wave >> 1);
  int ra[2], rb[TNW];  // of k-groups 0 and 1; those of 2 and 3 are turned by another 4 items
#pragma unroll
  for (int i = 0; i < 2; ++i) ra[i] = half * OA::KG + lds_row(wm + 32 * i + jl, half);
#pragma unroll
  for (int j = 0; j < TNW; ++j) rb[j] = OA::SIZE + half * OB::KG + lds_row(wn + 32 * j + jl, half);
  load_operand<TM, AL>(va, a.A, a.lda, m0, a.M, k_begin, k_end, tid);
  load_operand<TN, BL>(vb, a.B, a.ldb, n0, a.N, k_begin, k_end, tid);
  for (int k0 = k_begin; k0 < k_end; k0 += KC) {
    __syncthreads();
    store_operand<TM, AL>(s, va, tid);
    store_operand<TN, BL>(s + OA::SIZE, vb, tid);
    __syncthreads();
    if (k0 + KC < k_end) {
      load_operand<TM, AL>(va, a.A, a.lda, m0, a.M, k0 + KC, k_end, tid);
      load_operand<TN, BL>(vb, a.B, a.ldb, n0, a.N, k0 + KC, k_end, tid);
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      bf16x8 x[2][3];
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int i = 0; i < 2; ++i) x[i][q] = __builtin_bit_cast(bf16x8, s[(ra[i] ^ (4 * st)) + q * OA::TERM + 2 * st * OA::KG]);
#pragma unroll
      for (int j = 0; j < TNW; ++j) {
        bf16x8 y[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) y[q] = __builtin_bit_cast(bf16x8, s[(rb[j] ^ (4 * st)) + q * OB::TERM + 2 * st * OB::KG]);
        constexpr int P[6] = {2, 0, 1, 1, 0, 0}, Q[6] = {0, 2, 1, 0, 1, 0};  // the smallest products first
        if constexpr (SHORT) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            zr_f32x16 sum = {};
#pragma unroll
            for (int p = 0; p < 6; ++p) sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i][P[p]], y[Q[p]], sum, 0, 0, 0);
            acc[i][j] += sum;
            asm volatile("" : "+v"(acc[i][j]));  // done before the next sum: the registers hold no second one
          }
        } else {
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i)
              acc[i][j] = EPI == ZR_EPI_SOFTMAX_PARTIAL
                              ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i][P[p]], y[Q[p]], acc[i][j], 0, 0, 0)
                              : __builtin_amdgcn_mfma_f32_32x32x16_bf16(y[Q[p]], x[i][P[p]], acc[i][j], 0, 0, 0);
        }
      }
    }
  }

  bool finite = true;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TNW; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) finite = finite && fabsf(acc[i][j][r]) <= 3.402823466e38f;
  if (__any(!finite)) plain_tile<TNW, AL, BL, EPI == ZR_EPI_SOFTMAX_PARTIAL>(a, acc, m0 + wm, n0 + wn, k_begin, k_end, lane);

  if (EPI == ZR_EPI_STORE) {  // lane: row, register: column
    float* C = a.parts > 1 ? a.work + (long long)part * a.M * a.N : a.C;
    const long long ldc = a.parts > 1 ? a.M : a.ldc;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + wm + 32 * i + jl;
      const float b = (a.parts == 1 && a.bias && m < a.M) ? a.bias[m] : 0.0f;
#pragma unroll
      for (int j = 0; j < TNW; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int n = n0 + wn + 32 * j + 8 * (r >> 2) + 4 * half + (r & 3);
          if (m < a.M && n < a.N) {
            float* c = C + m + n * ldc;
            const float x = acc[i][j][r] + b;
            *c = (a.parts == 1 && a.accum) ? *c + x : x;
          }
        }
    }
  } else {  // lane: column, register: row; (max, sum exp) of every 32-row block and column
    const int nblocks = (a.M + 31) >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int mi = m0 + wm + 32 * i;
      const bool whole = mi + 32 <= a.M;
      float b[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = mi + 8 * (r >> 2) + 4 * half + (r & 3);
        b[r] = a.bias[m < a.M ? m : a.M - 1];
      }
#pragma unroll
      for (int j = 0; j < TNW; ++j) {
        const int n = n0 + wn + 32 * j + jl;
        float x[16], mx = -INFINITY, se = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[r] = acc[i][j][r] + b[r];
          if (whole || mi + 8 * (r >> 2) + 4 * half + (r & 3) < a.M) mx = fmaxf(mx, x[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (whole || mi + 8 * (r >> 2) + 4 * half + (r & 3) < a.M)
            se += __builtin_amdgcn_exp2f((x[r] - mx) * 1.4426950408889634f);
        se += __shfl_xor(se, 32, 64);
        if (n < a.N) {
          float* c = a.C + (long long)n * a.ldc + mi + 4 * half;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (whole) {
              *(f32x4u*)(c + 8 * q) = f32x4u{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (mi + 8 * q + 4 * half + e < a.M) c[8 * q + e] = x[4 * q + e];
            }
          }
          if (half == 0 && mi < a.M) {
            float* pp = a.partials + ((long long)n * nblocks + (mi >> 5)) * 2;
            pp[0] = mx;
            pp[1] = se;
          }
        }
      }
    }
  }
}

// C = the parts' sums, added in their order (+ bias, + C).
__global__ void __launch_bounds__(256) split_gemm_sum_kernel(SplitArgs a) {
  const long long mn = (long long)a.M * a.N;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < mn; i += (long long)gridDim.x * 256) {
    const int n = (int)(i / a.M), m = (int)(i - (long long)n * a.M);
    float x = a.work[i];
    for (int p = 1; p < a.parts; ++p) x += a.work[p * mn + i];
    if (a.bias) x += a.bias[m];
    float* c = a.C + m + n * a.ldc;
    *c = a.accum ? *c + x : x;
  }
}

template <int TNW, int AL, int BL>
void launch(const SplitArgs& a, unsigned grid, hipStream_t stream) {
  if (a.partials)
    split_gemm_kernel<TNW, AL, BL, ZR_EPI_SOFTMAX_PARTIAL><<<grid, 256, 0, stream>>>(a);
  else
    split_gemm_kernel<TNW, AL, BL, ZR_EPI_STORE><<<grid, 256, 0, stream>>>(a);
}

template <int TNW>
void launch_layouts(const SplitArgs& a, int al, int bl, unsigned grid, hipStream_t stream) {
  if (al == ZR_SPLIT_PACK4)
    launch<TNW, ZR_SPLIT_PACK4, ZR_SPLIT_K_FAST>(a, grid, stream);
  else if (al == ZR_SPLIT_K_FAST && bl == ZR_SPLIT_K_FAST)
    launch<TNW, ZR_SPLIT_K_FAST, ZR_SPLIT_K_FAST>(a, grid, stream);
  else if (al == ZR_SPLIT_K_FAST)
    launch<TNW, ZR_SPLIT_K_FAST, ZR_SPLIT_ROW_FAST>(a, grid, stream);
  else if (bl == ZR_SPLIT_K_FAST)
    launch<TNW, ZR_SPLIT_ROW_FAST, ZR_SPLIT_K_FAST>(a, grid, stream);
  else
    launch<TNW, ZR_SPLIT_ROW_FAST, ZR_SPLIT_ROW_FAST>(a, grid, stream);
}

}  // namespace

int zr_split_gemm(zr_ctx* ctx, int M, int N, int K, const float* A, long long lda, int a_layout, const float* B,
                  long long ldb, int b_layout, float* C, long long ldc, const float* bias, float* partials, int accumulate) {
  ZR_CHECK_ARG(b_layout != ZR_SPLIT_PACK4 && (a_layout != ZR_SPLIT_PACK4 || b_layout == ZR_SPLIT_K_FAST),
               "split product: operand layouts %d, %d", a_layout, b_layout);
  SplitArgs a = {};
  a.M = M, a.N = N, a.K = K;
  a.A = A, a.lda = lda, a.B = B, a.ldb = ldb, a.C = C, a.ldc = ldc;
  a.bias = bias, a.partials = partials, a.accum = accumulate;
  a.m_tiles = (M + TM - 1) / TM;
  const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  // K in parts where the tiles alone would leave compute units idle, each part's sums to scratch and added in order.
  // No parts without scratch to be had: the fixed buffers are not for this, and nothing may be allocated under capture.
  size_t most = 192u << 20;
  if (partials || ctx->fixed_scratch) {
    most = 0;
  } else {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &capture) != hipSuccess) (void)hipGetLastError();
    if (capture != hipStreamCaptureStatusNone && ctx->scratch_bytes < most) most = ctx->scratch_bytes;
  }
  int tnw = 2;
  double best = 0.0;
  for (int w = 2; w <= 4; w += 2) {
    const long long tiles = (long long)a.m_tiles * ((N + 64 * w - 1) / (64 * w));
    for (int p = 1; p <= 64; ++p) {
      const size_t bytes = sizeof(float) * (size_t)M * N * p;
      if (p > 1 && (K < p * 4 * KC || bytes > most)) break;
      const double us = zr_split_launch_us(w, tiles * p, (K + p * KC - 1) / (p * KC), cus) + (p > 1 ? 6.0 + (double)bytes / 4.0e6 : 0.0);
      if (best == 0.0 || us < best) best = us, tnw = w, a.parts = p;
    }
  }
  a.n_tiles = (N + 64 * tnw - 1) / (64 * tnw);
  a.k_part = ((K + a.parts - 1) / a.parts + KC - 1) / KC * KC;
  a.parts = (K + a.k_part - 1) / a.k_part;
  if (a.parts > 1) {
    void* p = nullptr;
    const int rc = zr_ctx_scratch(ctx, 0, sizeof(float) * (size_t)M * N * a.parts, &p);
    if (rc) return rc;
    a.work = (float*)p;
  }
  const unsigned grid = (unsigned)(((long long)a.m_tiles * a.n_tiles * a.parts + 7) / 8 * 8);
  if (tnw == 4)
    launch_layouts<4>(a, a_layout, b_layout, grid, ctx->stream);
  else
    launch_layouts<2>(a, a_layout, b_layout, grid, ctx->stream);
  ZR_LAUNCH_CHECK("split_gemm_kernel");
  if (a.parts > 1) {
    const long long blocks = ((long long)M * N + 255) / 256;
    split_gemm_sum_kernel<<<(unsigned)(blocks < 4096 ? blocks : 4096), 256, 0, ctx->stream>>>(a);
    ZR_LAUNCH_CHECK("split_gemm_sum_kernel");
  }
  return ZR_OK;
}
