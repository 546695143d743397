// The output layer's product on a prepared bf16 matrix for up to 64 columns, with the soft-max partials.
//
// A wave owns 32 rows and all columns: its part of the matrix goes from memory straight to its registers, two chunks of 64 k ahead, once in the launch.
// The activations, split into bf16 terms beforehand, go through LDS, as far ahead, with loads that write LDS directly.  Workgroups of four waves, so that
// several share a compute unit and one's loads fly beside another's products.
// gemm_rows_kernel's workgroups split K over their waves instead: a sum through LDS for every few rows, no loads in flight meanwhile.
// Four accumulators an output (terms, and steps of 16 k in turn), so that no chain is longer than there.
// Bound: the matrix's way from memory at a few columns (8: 105 MB past L2 at 5.2 TB/s); at 37 and 64 neither memory (4.5 and 4.2 TB/s) nor the matrix pipes (busy
// for a quarter) are full, the waits at the steps' barriers are left.  50000 x 1024, us of a call: 64 columns 36.1 -> 30.7, 37 34.8 -> 27.0, 8 22.1 -> 20.8.  Three chunks
// ahead instead of two measured the same.
#include "zr_internal.h"
#include "zr_logits_epilogue.h"
#include "zr_mfma_core.h"

namespace {

constexpr int W = 4;        // waves a workgroup
constexpr int CG = 8;       // k-groups of 8 a chunk
constexpr int STEPS = CG / 2;

struct Logits16Args {
  int M, N, K, ldp;
  const unsigned short* A;          // [K/8][ldp][8]
  const unsigned short *hi, *lo;    // [K/8][N][8]
  float* C;
  long long ldc;
  const float* bias;
  float* partials;
};

template <int TN, bool LO, int WAUX>
__global__ void __launch_bounds__(64 * W, 2) logits_bf16_kernel(Logits16Args a) {
  constexpr int COLS = 32 * TN, NT = LO ? 2 : 1, NACC = 4;
  constexpr int BUF = NT * CG * COLS;              // 16-byte elements of a chunk: [term][k-group][column]
  constexpr int NI = BUF / (64 * W);               // of a thread
  __shared__ zr_u32x4 s0[BUF], s1[BUF], s2[BUF];   // three arrays: the compiler sees that a read of one need not wait for loads into another
  const int tid = threadIdx.x, lane = tid & 63, jl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = ((int)blockIdx.x * W + wave) * 32;
  const int row = m0 + jl < a.M ? m0 + jl : a.M - 1;
  const int kgroups = a.K >> 3, chunks = (kgroups + CG - 1) / CG;
  // Both operands through descriptors that end at k = K: the last chunk reads zeros behind it.
  const unsigned kstep = 16u * (unsigned)a.ldp, xstep = 16u * (unsigned)a.N;
  const __amdgpu_buffer_rsrc_t arsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.A), 0, (int)((unsigned)kgroups * kstep), 0x00020000);
  const __amdgpu_buffer_rsrc_t hrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.hi), 0, (int)((unsigned)kgroups * xstep), 0x00020000);
  const __amdgpu_buffer_rsrc_t lrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(LO ? a.lo : a.hi), 0, (int)((unsigned)kgroups * xstep), 0x00020000);
  const unsigned aoff = 16u * (unsigned)row + (unsigned)half * kstep;
  auto load_a = [&](zr_u32x4 (&v)[STEPS], int c) {
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
      v[st] = __builtin_amdgcn_raw_buffer_load_b128(arsrc, (int)(aoff + (unsigned)(c * CG + 2 * st) * kstep), 0, WAUX);
  };
  auto load_x = [&](int c, zr_u32x4* s) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int item = tid + 64 * W * i, kg = item / COLS % CG, col = item % COLS;  // (a term's items are a multiple of the workgroup)
      const unsigned off = (unsigned)(c * CG + kg) * xstep + 16u * (unsigned)(col < a.N ? col : a.N - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < NI / NT ? hrsrc : lrsrc,
                                               (__attribute__((address_space(3))) void*)(s + i * 64 * W + wave * 64), 16, (int)off, 0, 0, 0);
    }
  };
  zr_f32x16 acc[NACC][TN];
#pragma unroll
  for (int q = 0; q < NACC; ++q)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[q][j][r] = 0.0f;
  auto compute = [&](const zr_u32x4 (&v)[STEPS], const zr_u32x4* s) {
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int q = LO ? 2 * (st & 1) + t : st;
          const zr_u32x4 x = s[(t * CG + 2 * st + half) * COLS + 32 * j + jl];
          acc[q][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(zr_bf16x8, v[st]), __builtin_bit_cast(zr_bf16x8, x), acc[q][j], 0, 0, 0);
        }
  };
  zr_u32x4 ar0[STEPS], ar1[STEPS], ar2[STEPS];
  // Chunk c: its activations have landed in every wave's part once the loads asked for behind them (a chunk's activations and matrix, less what the
  // products wait for anyway) are all that is in flight.  The buffer that is filled next was last read in chunk c - 1, behind the barrier.
  auto step = [&](int c, const zr_u32x4 (&v)[STEPS], const zr_u32x4* x, zr_u32x4 (&vn)[STEPS], zr_u32x4* xn) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (NI + STEPS));  // vmcnt
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");  // nothing behind the barrier is read before it (a fence would wait for every load)
    __builtin_amdgcn_sched_barrier(0);
    load_x(c + 2, xn);
    load_a(vn, c + 2);
    __builtin_amdgcn_sched_barrier(0);
    compute(v, x);
    __builtin_amdgcn_sched_barrier(0);
  };
  load_x(0, s0);
  load_a(ar0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load_x(1, s1);
  load_a(ar1, 1);
  __builtin_amdgcn_sched_barrier(0);
  for (int c = 0; c < chunks; c += 3) {  // (chunks behind the last one are zeros)
    step(c, ar0, s0, ar2, s2);
    step(c + 1, ar1, s1, ar0, s0);
    step(c + 2, ar2, s2, ar1, s1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // no load into LDS outlives the workgroup
  if (m0 >= a.M) return;
#pragma unroll
  for (int j = 0; j < TN; ++j) acc[0][j] = (acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j]);
  zr_logits_epilogue<TN>(acc[0], m0, 0, a.M, a.N, a.C, a.ldc, a.bias, a.partials, lane);
}

template <int TN, bool LO>
void launch(const Logits16Args& a, bool stream, hipStream_t st) {
  const unsigned grid = (unsigned)((a.M + 32 * W - 1) / (32 * W));
  if (stream)
    logits_bf16_kernel<TN, LO, ZR_AUX_STREAM><<<grid, 64 * W, 0, st>>>(a);
  else
    logits_bf16_kernel<TN, LO, 0><<<grid, 64 * W, 0, st>>>(a);
}

}  // namespace

int zr_logits_bf16(zr_ctx* ctx, int V, int cols, int H, const unsigned short* packed, int ldp, const unsigned short* hi, const unsigned short* lo, float* C,
                   long long ldc, const float* bias, float* partials, bool stream) {
  const Logits16Args a = {V, cols, H, ldp, packed, hi, lo, C, ldc, bias, partials};
  if (cols <= 32)
    lo ? launch<1, true>(a, stream, ctx->stream) : launch<1, false>(a, stream, ctx->stream);
  else
    lo ? launch<2, true>(a, stream, ctx->stream) : launch<2, false>(a, stream, ctx->stream);
  ZR_LAUNCH_CHECK("logits_bf16_kernel");
  return ZR_OK;
}
