// The output layer's product on a prepared fp32 matrix for up to 16 columns -- one sentence's beam, the width the reference decodes
// at -- with the soft-max partials: a stream of the matrix through the chip, 200 MB for 1.2 GFLOP at 50000 x 1000 x 12.
//
// A wave owns 32 rows and all columns on the 16 x 16 x 4 instruction, whose operands are one 16-byte load a lane for 16 k in the k-interleaved
// layout, five groups of 16 k ahead.  Waves are workgroups of their own, so that they spread evenly over the compute units, or four of them
// with 64 rows each (1 KB of neighbouring memory a k-block; zr_logits_narrow_pairs).  32 x 32 x 2 instructions leave more than half of their columns empty at this
// width: 30 us of them in a row at 50000 x 1000, on one wave a SIMD, beside 41 us for the launch that had them.  The activations are read as they lie.  No LDS, no barrier.
// Bound: the matrix's way from memory, 6.3 TB/s.  That launch with its re-layout of the activations where needed / this one, us: 50000 x 1000 x 12 40.4 -> 31.8,
// 50000 x 500 33.1 -> 17.3, 30000 x 1000 38.2 -> 18.8, 30011 x 333 x 10 (K % 8 != 0, another kernel) 15.1 -> 7.8, 10000 x 100 x 8 7.8 -> 4.8.  More groups in
// flight (six, eight) 1 to 5 % slower.  Mean error against 64 bits with eight sums an output, with two, and before, 1e-9: H = 300 3.8, 6.2, 4.8; 500 5.9, 10.2, 7.7;
// 1000 11, 20, 27: the same time.
#include "zr_internal.h"
#include "zr_mfma_core.h"

namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any multiple of 4

struct NarrowArgs {
  int M, N, K, ldp, kp;  // A: element (row, k) at ((k/4)*ldp + row)*4 + k%4, k < kp
  const float* A;
  const float* B;        // column n at n*ldb
  long long ldb;
  float* C;
  long long ldc;
  const float* bias;
  float* partials;
};

// TM: 32-row blocks a wave.  PF: groups of 16 k in flight.
template <int TM, int PF, int W, int WAUX>
__global__ void __launch_bounds__(64 * W, 2) logits_narrow_kernel(NarrowArgs a) {
  constexpr int T = 2 * TM;  // 16-row tiles
  constexpr int NA = 8;      // sums an output, in turn over k: the shorter they are the less they round
  const int lane = threadIdx.x & 63, cl = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * W + (threadIdx.x >> 6)));
  const int m0 = 32 * TM * wave;
  if (m0 >= a.M) return;
  const int groups = (a.K + 15) >> 4;
  // What lies past the matrix's last k-block, and past its last row block, reads as zero.
  const __amdgpu_buffer_rsrc_t arsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.A), 0, (int)(unsigned)((long long)a.kp * a.ldp * 4), 0x00020000);
  const unsigned kstep = 16u * (unsigned)a.ldp;  // bytes of four k
  unsigned off[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int row = m0 + 16 * t + cl;
    off[t] = 16u * (unsigned)(row < a.ldp ? row : a.ldp - 1) + (unsigned)kq * kstep;
  }
  const float* col = a.B + (long long)(cl < a.N ? cl : a.N - 1) * a.ldb;
  struct Frag {
    zr_f32x4 w[T], x;
  };
  Frag f[PF + 1];
  auto load = [&](Frag& q, int g) {
#pragma unroll
    for (int t = 0; t < T; ++t)
      q.w[t] = __builtin_bit_cast(zr_f32x4, __builtin_amdgcn_raw_buffer_load_b128(arsrc, (int)off[t], (int)(4u * (unsigned)g * kstep), WAUX));
    const int k0 = 16 * g + 4 * kq, ks = k0 < a.K - 4 ? k0 : a.K - 4;
    q.x = *(const f32x4u*)(col + ks);
  };
  zr_f32x4 acc[NA][T];
#pragma unroll
  for (int q = 0; q < NA; ++q)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[q][t] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto mma = [&](Frag& q, int g, int first) {
    if (16 * (g + 1) > a.K) {  // the columns end inside this group: shift the moved load back, zero what lies behind
      const int d = 16 * g + 4 * kq - (a.K - 4);
      const zr_f32x4 v = q.x;
      if (d > 0) {
        q.x[0] = d == 1 ? v[1] : (d == 2 ? v[2] : (d == 3 ? v[3] : 0.0f));
        q.x[1] = d == 1 ? v[2] : (d == 2 ? v[3] : 0.0f);
        q.x[2] = d == 1 ? v[3] : 0.0f;
        q.x[3] = 0.0f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < T; ++t) acc[first + e][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(q.w[t][e], q.x[e], acc[first + e][t], 0, 0, 0);
  };
  const int last = groups - 1;
#pragma unroll
  for (int s = 0; s < PF; ++s) load(f[s], s < last ? s : last);
  int g = 0;
  for (; g + PF + 1 <= groups; g += PF + 1) {
#pragma unroll
    for (int s = 0; s < PF + 1; ++s) {
      load(f[(s + PF) % (PF + 1)], g + s + PF < last ? g + s + PF : last);
      mma(f[s], g + s, (s & 1) * 4);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int s = 0; s < PF; ++s)
    if (g + s < groups) mma(f[s], g + s, (s & 1) * 4);

  // A lane has one column and rows 4 kq .. 4 kq + 3 of every 16-row tile.
  const int nblocks = (a.M + 31) >> 5;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int mb = m0 + 32 * b;
    if (mb >= a.M) break;
    float x[2][4], mx = -INFINITY, se = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mb + 16 * h + 4 * kq + r;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < NA; q += 2) v += acc[q][2 * b + h][r] + acc[q + 1][2 * b + h][r];
        x[h][r] = v + a.bias[m < a.M ? m : a.M - 1];
        if (m < a.M) mx = fmaxf(mx, x[h][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (mb + 16 * h + 4 * kq + r < a.M) se += __builtin_amdgcn_exp2f((x[h][r] - mx) * 1.4426950408889634f);
    se += __shfl_xor(se, 16, 64);
    se += __shfl_xor(se, 32, 64);
    if (cl >= a.N) continue;
    float* c = a.C + (long long)cl * a.ldc + mb + 4 * kq;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (mb + 32 <= a.M) {
        *(f32x4u*)(c + 16 * h) = f32x4u{x[h][0], x[h][1], x[h][2], x[h][3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (mb + 16 * h + 4 * kq + r < a.M) c[16 * h + r] = x[h][r];
      }
    }
    if (kq == 0) {
      float* pp = a.partials + ((long long)cl * nblocks + (mb >> 5)) * 2;
      pp[0] = mx;
      pp[1] = se;
    }
  }
}

template <int TM, int PF, int W>
void launch(const NarrowArgs& a, bool stream, hipStream_t st) {
  const unsigned grid = (unsigned)((a.M + 32 * W * TM - 1) / (32 * W * TM));
  if (stream)
    logits_narrow_kernel<TM, PF, W, ZR_AUX_STREAM><<<grid, 64 * W, 0, st>>>(a);
  else
    logits_narrow_kernel<TM, PF, W, 0><<<grid, 64 * W, 0, st>>>(a);
}

}  // namespace

int zr_logits_narrow(zr_ctx* ctx, int V, int cols, int H, const float* packed, int ldp, const float* h, long long ldh, float* C, long long ldc,
                     const float* bias, float* partials, bool stream) {
  const NarrowArgs a = {V, cols, H, ldp, (H + 7) / 8 * 8, packed, h, ldh, C, ldc, bias, partials};
  if (zr_logits_narrow_pairs(V, H, ctx->cu_count))
    launch<2, 4, 4>(a, stream, ctx->stream);
  else
    launch<1, 4, 1>(a, stream, ctx->stream);
  ZR_LAUNCH_CHECK("logits_narrow_kernel");
  return ZR_OK;
}
