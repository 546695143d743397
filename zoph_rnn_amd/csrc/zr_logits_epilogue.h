// Behind an output-layer product of 32 x 32 blocks with the weights first: logits and the soft-max partials, shared by the kernels on fp32 and on bf16
// matrices.
#pragma once
#include "zr_internal.h"

typedef float zr_f32x4_any __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any multiple of 4

// One wave's 32 rows from m0 on (m0 < M) of TN blocks of 32 columns from n0 on.
template <int TN>
__device__ __forceinline__ void zr_logits_epilogue(const zr_f32x16 (&acc)[TN], int m0, int n0, int M, int N, float* C, long long ldc, const float* bias,
                                                   float* partials, int lane) {
  const int jl = lane & 31, half = lane >> 5;
  // A lane has one column of each 32 x 32 block and sixteen of its rows: logits, and (max, sum exp) of the block's column.
  const int nblocks = (M + 31) >> 5;
  const bool whole = m0 + 32 <= M;
  float b[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + 8 * (r >> 2) + 4 * half + (r & 3);
    b[r] = bias[m < M ? m : M - 1];
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + 32 * j + jl;
    float x[16], mx = -INFINITY, se = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      x[r] = acc[j][r] + b[r];
      if (whole || m0 + 8 * (r >> 2) + 4 * half + (r & 3) < M) mx = fmaxf(mx, x[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (whole || m0 + 8 * (r >> 2) + 4 * half + (r & 3) < M) se += __builtin_amdgcn_exp2f((x[r] - mx) * 1.4426950408889634f);
    se += __shfl_xor(se, 32, 64);
    if (n < N) {
      float* c = C + (long long)n * ldc + m0 + 4 * half;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (whole) {
          *(zr_f32x4_any*)(c + 8 * q) = zr_f32x4_any{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (m0 + 8 * q + 4 * half + e < M) c[8 * q + e] = x[4 * q + e];
        }
      }
      if (half == 0) {
        float* pp = partials + ((long long)n * nblocks + (m0 >> 5)) * 2;
        pp[0] = mx;
        pp[1] = se;
      }
    }
  }
}
