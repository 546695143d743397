// Folding of the output layer's per-32-row-block (max, sum exp(x - max)) pairs into one pair per column: shared by
// the kernels that normalise (zr_softmax.hip) and the beam's selection on blocks (zr_beam.hip), so that all arrive at the
// same bits (outputdist_overflow_prevention_kernel, src/custom_kernels.h:503-577, takes one max and one sum per column;
// here they are assembled from the blocks in one fixed order).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

// All 256 threads of a workgroup call this with the column's pairs ([nblocks][2] floats, contiguous) and have the column's (max,
// sum) on return.  The maximum first, then every block's sum scaled to it once: one exponential a pair, where a running pair
// takes two for every pair and for every step of the butterfly.  (expf: in a column with all blocks a distance d below one large logit the
// errors have one sign, and exp2 of a rounded d * log2 e is off by d * 2^-24.)  `behind_loads` is called once the first 2048 pairs are on
// their way; returns the largest block maximum this thread saw (-inf if none).  s_m, s_s: four floats of shared memory each.
template <class F>
__device__ __forceinline__ float zr_softmax_fold_column(const float* __restrict__ pairs, int nblocks, float* s_m, float* s_s,
                                                        float& mx, float& sum, F&& behind_loads) {
  typedef float zr_f32x2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const zr_f32x2* pp = (const zr_f32x2*)pairs;
  zr_f32x2 pr[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int b = tid + 256 * u;
    pr[u] = zr_f32x2{-INFINITY, 0.0f};
    if (b < nblocks) pr[u] = pp[b];
  }
  behind_loads();
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < 8; ++u) m = fmaxf(m, pr[u].x);  // (NaN never wins a maximum)
  for (int b = tid + 2048; b < nblocks; b += 256) m = fmaxf(m, pp[b].x);
  const float mine = m;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if (lane == 0) s_m[wave] = m;
  __syncthreads();
  mx = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
  // (a block at the maximum counts as it is: also where both are infinite)
  auto scaled = [&](const zr_f32x2& p) { return p.x == mx ? p.y : p.y * expf(p.x - mx); };
  float s = 0.0f;
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (256 * u < nblocks) s += scaled(pr[u]);  // uniform
  for (int b = tid + 2048; b < nblocks; b += 256) s += scaled(pp[b]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) s_s[wave] = s;
  __syncthreads();
  sum = (s_s[0] + s_s[1]) + (s_s[2] + s_s[3]);
  return mine;
}
