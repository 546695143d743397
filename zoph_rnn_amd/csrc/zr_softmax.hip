// Output softmax: logits on MFMA (bias and per-32-row (max, sum exp) partials fused into the GEMM epilogue),
// then one read + one write of the V x mb matrix to normalise.
#include <math.h>

#include "zr_internal.h"
#include "zr_softmax_fold.h"

namespace {

// Folds the per-32-row partials of one column ([N][nblocks][2] floats: contiguous per column, nblocks
// (max, sum exp(x - max)) pairs) into the column's (max, sum).  One workgroup per column (zr_softmax_fold.h).
__global__ void __launch_bounds__(256)
softmax_colstats_kernel(const float* __restrict__ partials, int nblocks, float* __restrict__ colstats) {
  __shared__ float s_m[4], s_s[4];
  const int n = blockIdx.x;
  float mx, sum;
  zr_softmax_fold_column(partials + (size_t)n * nblocks * 2, nblocks, s_m, s_s, mx, sum, [] {});
  if (threadIdx.x == 0) {
    colstats[2 * n] = mx;
    colstats[2 * n + 1] = sum;
  }
}

// out = exp(x - max) / sum   (MODE 0)   or   (x - max) - log(sum)   (MODE 1); in and out may be the same matrix.  A
// workgroup takes 1024 * U rows of one column, U 16-byte accesses a thread at any alignment.  FOLD: it folds the column's block pairs itself,
// while its logits are on their way, which saves the launch of softmax_colstats_kernel; else `pairs` holds that one's statistics.
// Both launches before / this one, us: 10000 x 8 6.0 -> 2.8, 30011 x 37 (odd columns had 4-byte accesses) 8.9 -> 5.7, 40000 x 64 11.6 -> 10.8,
// 30000 x 128 14.3 -> 10.2.  Bound by memory from there on, with the statistics in a launch of their own: 50000 x 128 15.4 us, the fold by every workgroup 16.4; 80000 x 256
// 29.6 and 34.5; 80001 x 256 41.4 -> 30.1 by the accesses' width.
template <int MODE, int U, bool FOLD>
__global__ void __launch_bounds__(256)
softmax_normalize_kernel(const float* in, float* out, int V, const float* __restrict__ pairs, int nblocks) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  __shared__ float s_m[4], s_s[4];
  const int n = blockIdx.y;
  const float* x = in + (size_t)n * V;
  float* y = out + (size_t)n * V;
  const int first = (blockIdx.x * U * 256 + threadIdx.x) * 4;
  f32x4u v[U];
  auto load = [&] {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = first + 1024 * u;
      if (i + 4 <= V) {
        v[u] = *(const f32x4u*)(x + i);
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (i + e < V) v[u][e] = x[i + e];
      }
    }
  };
  float mx, sum;
  if constexpr (FOLD) {
    zr_softmax_fold_column(pairs + (size_t)n * nblocks * 2, nblocks, s_m, s_s, mx, sum, load);
  } else {
    mx = pairs[2 * n], sum = pairs[2 * n + 1];
    load();
  }
  const float lsum = MODE == 1 ? logf(sum) : 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = first + 1024 * u;
    f32x4u r;
#pragma unroll
    for (int e = 0; e < 4; ++e)  // expf(x - max) / sum, as the reference divides (custom_kernels.h:574-576)
      r[e] = MODE == 0 ? expf(v[u][e] - mx) / sum : (v[u][e] - mx) - lsum;
    if (i + 4 <= V) {
      *(f32x4u*)(y + i) = r;
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (i + e < V) y[i + e] = r[e];
    }
  }
}

// x (V x n logits) -> e = onehot(target) - p in place, p = exp(x - max) / sum as softmax_normalize_kernel has it, 0 on masked
// columns; the sums of e over the workgroup's `cols` columns to sums[blockIdx.y][V], and every column's target probability.  The three readers of the probabilities (errors, gradient of the bias, loss) were passes of their own over
// the matrix: at 50000 x 6400 normalise 483, error 499, bias sums 250 us, bound by memory; this pass reads and writes once.
// VEC: four consecutive rows per thread with 16-byte accesses (V % 4 == 0, x and sums 16-byte aligned).
template <bool VEC>
__global__ void __launch_bounds__(256)
softmax_error_kernel(float* __restrict__ x, int V, int n, int cols, const float* __restrict__ colstats, const int* __restrict__ target,
                     const int* __restrict__ mask01, float* __restrict__ sums, float* __restrict__ p_target) {
  constexpr int W = VEC ? 4 : 1;
  typedef float vec __attribute__((ext_vector_type(W)));
  const int v = (blockIdx.x * 256 + threadIdx.x) * W;
  if (v >= V) return;
  const int n0 = blockIdx.y * cols, n1 = min(n, n0 + cols);
  vec s = {};
#pragma unroll 4
  for (int c = n0; c < n1; ++c) {
    vec* q = (vec*)(x + (size_t)c * V + v);
    const vec in = *q;
    const float mx = colstats[2 * c], sum = colstats[2 * c + 1];
    const bool on = mask01[c] == 1;
    const int tg = min(max(target[c], 0), V - 1);
    vec e;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const float p = expf(in[i] - mx) / sum;
      if (v + i == tg) p_target[c] = p;
      e[i] = on ? (v + i == target[c] ? 1.0f : 0.0f) - p : 0.0f;
    }
    *q = e;
    s += e;
  }
  *(vec*)(sums + (size_t)blockIdx.y * V + v) = s;
}

// Double-precision column statistics (outputdist_perplexity_kernel accumulates in double, reference:
// src/custom_kernels.h:583-660).  The column's largest logit comes from the product's block pairs, whose maxima are of the
// very values it stored, so the logits are read once, and are on their way while the pairs are folded.  gridDim.y workgroups
// share a column: one (colstats = max, log sum) unless the columns alone would leave compute units idle; of several each
// leaves its part of the sum in sums[column][part].
// Bound by the logits' way from memory and the 64-bit exponentials together.  700 columns of 33333: 89 us with two passes of
// single loads by 256 threads, 32 us so.
constexpr int kF64Threads = 512;
__global__ void __launch_bounds__(kF64Threads)
softmax_colstats_f64_kernel(const float* __restrict__ logits, int V, const float* __restrict__ pairs, int nblocks, double* __restrict__ colstats,
                            double* __restrict__ sums) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  constexpr int WAVES = kF64Threads / 64, U = 4, SPAN = 4 * kF64Threads;
  __shared__ float s_m[WAVES];
  __shared__ double s_s[WAVES];
  const int n = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* x = logits + (size_t)n * V;
  const int share = (V / 4 + (int)gridDim.y - 1) / (int)gridDim.y * 4;  // the last workgroup also takes the V % 4 left over
  const int begin = min((int)blockIdx.y * share, V), end = blockIdx.y + 1 == gridDim.y ? V : min(begin + share, V);
  f32x4u v[U];
  auto load = [&](int at) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = at + 4 * tid + SPAN * u;
      v[u] = f32x4u{-INFINITY, -INFINITY, -INFINITY, -INFINITY};  // adds exp(-inf) = 0
      if (i + 4 <= end) {
        v[u] = *(const f32x4u*)(x + i);
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (i + e < end) v[u][e] = x[i + e];
      }
    }
  };
  load(begin);
  float m = -INFINITY;
  const f32x2* pp = (const f32x2*)(pairs + (size_t)n * nblocks * 2);
  for (int b = tid; b < nblocks; b += kF64Threads) m = fmaxf(m, pp[b].x);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if (lane == 0) s_m[wave] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) m = fmaxf(m, s_m[w]);
  const double mx = fmax(-1.7976931348623157e308, (double)m);
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  for (int at = begin; at < end; at += SPAN * U) {
    f32x4u now[U];
#pragma unroll
    for (int u = 0; u < U; ++u) now[u] = v[u];
    if (at + SPAN * U < end) load(at + SPAN * U);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (at + 4 * tid + SPAN * u >= end) break;  // (nothing but zeros: small vocabularies)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] += exp((double)now[u][e] - mx);
    }
  }
  double total = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off, 64);
  if (lane == 0) s_s[wave] = total;
  __syncthreads();
  if (tid != 0) return;
  total = 0.0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) total += s_s[w];
  if (blockIdx.y == 0) colstats[2 * n] = mx;
  if (gridDim.y == 1)
    colstats[2 * n + 1] = log(total);
  else
    sums[(size_t)n * gridDim.y + blockIdx.y] = total;
}

__global__ void __launch_bounds__(256)
softmax_logprob_f64_kernel(const float* __restrict__ logits, double* __restrict__ out, int V,
                           const double* __restrict__ colstats) {
  const int n = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < V) out[(size_t)n * V + i] = ((double)logits[(size_t)n * V + i] - colstats[2 * n]) - colstats[2 * n + 1];
}

// loss = sum over unmasked columns of log p[target[b], b]; single workgroup, fixed summation order.  parts: workgroups of
// softmax_colstats_f64_kernel that shared a column.
__global__ void __launch_bounds__(256)
softmax_loss_kernel(const float* __restrict__ logits, int V, int mb, const double* __restrict__ colstats, const double* __restrict__ sums, int parts,
                    const int* __restrict__ target, const int* __restrict__ mask01, double* __restrict__ loss,
                    int* __restrict__ flags) {
  __shared__ double s[256];
  const int tid = threadIdx.x;
  double acc = 0.0;
  for (int b = tid; b < mb; b += 256) {
    if (mask01[b] == 1) {
      int t = target[b];
      if (t < 0 || t >= V) {
        atomicAdd(&flags[0], 1);
        t = t < 0 ? 0 : V - 1;
      }
      double lsum = colstats[2 * b + 1];
      if (parts > 1) {
        lsum = 0.0;
        for (int q = 0; q < parts; ++q) lsum += sums[(size_t)b * parts + q];
        lsum = log(lsum);
      }
      acc += ((double)logits[(size_t)b * V + t] - colstats[2 * b]) - lsum;
    }
  }
  s[tid] = acc;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (tid < st) s[tid] += s[tid + st];
    __syncthreads();
  }
  if (tid == 0) loss[0] = s[0];
}

template <int MODE>
int launch_normalize(zr_ctx* ctx, const float* in, float* out, int V, int mb, const float* pairs, int nblocks, float* colstats) {
  const ZrNormalizePlan plan = zr_softmax_normalize_plan(V, mb);
  const dim3 grid((V + 1024 * plan.accesses - 1) / (1024 * plan.accesses), mb);
  if (!plan.fold) {
    const int rc = zr_softmax_colstats_launch(ctx, pairs, nblocks, mb, colstats);
    if (rc) return rc;
    softmax_normalize_kernel<MODE, 2, false><<<grid, 256, 0, ctx->stream>>>(in, out, V, colstats, nblocks);
  } else if (plan.accesses == 1) {
    softmax_normalize_kernel<MODE, 1, true><<<grid, 256, 0, ctx->stream>>>(in, out, V, pairs, nblocks);
  } else if (plan.accesses == 2) {
    softmax_normalize_kernel<MODE, 2, true><<<grid, 256, 0, ctx->stream>>>(in, out, V, pairs, nblocks);
  } else {
    softmax_normalize_kernel<MODE, 4, true><<<grid, 256, 0, ctx->stream>>>(in, out, V, pairs, nblocks);
  }
  ZR_LAUNCH_CHECK("softmax_normalize_kernel");
  return ZR_OK;
}

// d_h_packed: optional k-interleaved copy of d_h ([H/4][mb][4]); used when the product runs on the registered fp32 copy
// of D and H % 8 == 0 (the product then skips its own re-layout of d_h), but not where zr_logits_plan or the split product
// takes the call, which read d_h as it lies: with and without the copy the same kernel runs.
// d_partials_ext: where the [mb][nblocks][2] pairs go instead of context scratch (ZR_SOFTMAX_LOGITS_BLOCKS: the caller's
// buffer; no column statistics follow them there).
int logits_with_partials(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb,
                         float* d_logits, float** partials_out, int* nblocks_out, const float* d_h_packed = nullptr,
                         const unsigned short* d_h_hi = nullptr, const unsigned short* d_h_lo = nullptr,
                         float* d_partials_ext = nullptr) {
  const int nblocks = zr_softmax_partial_blocks(V);
  void* scratch = d_partials_ext;
  int rc = ZR_OK;
  if (!scratch) {
    // partials [mb][nblocks][2] followed by column stats (2 doubles per column, also used as 2 floats)
    const size_t pbytes = sizeof(float) * 2 * (size_t)nblocks * mb;
    rc = zr_ctx_scratch(ctx, 1, pbytes + sizeof(double) * 2 * (size_t)mb + 64, &scratch);
    if (rc) return rc;
  }
  ZrGemmDesc d = {};
  d.M = V;
  d.N = mb;
  d.nseg = 1;
  d.K[0] = H;
  d.A[0] = d_D;
  d.lda[0] = V;
  ZrLogitsPlan plan = {0, 0};
  for (int i = 0; i < ZR_MAX_PACKED_D; ++i) {
    const zr_ctx::PackedD& e = ctx->packed_d[i];
    if (e.key == d_D && e.V == V && e.H == H) {  // registered with zr_softmax_prepare: use the MFMA-layout copy
      if (!e.bf16 && ctx->gemm_cfg == 0) plan = zr_logits_plan(V, mb, H, ctx->cu_count);
      // ... unless the batch is thousands of columns wide (all time steps of a training minibatch at once) and that kernel does
      // not take it: there the split terms, which read either form, or the LDS-staged kernel on the plain matrix are faster than
      // the register-streaming one on the fp32 copy
      if (!e.bf16 && mb > 1024 && !plan.tn) break;
      d.A[0] = (const float*)e.d_pack;
      d.lda[0] = e.ldp;
      d.a_pack = e.bf16 ? 2 : 1;
      break;
    }
  }
  const bool stream = (size_t)V * H * (d.a_pack == 2 ? 2 : 4) >= ((size_t)64 << 20);
  const bool narrow = d.a_pack == 1 && ctx->gemm_cfg == 0 && zr_logits_narrow_takes(V, mb, H);
  if (plan.tn || narrow) {
    if (ctx->fixed_scratch && mb <= 1024 && V >= 2048 && H % 8 == 0 && ((uintptr_t)d_h & 15u) == 0) {
      // nothing of it is used here; the limit of the entry point does not follow the kernel
      void* p = nullptr;
      rc = zr_ctx_scratch(ctx, 0, sizeof(float) * (size_t)H * mb, &p);
      if (rc) return rc;
    }
    rc = narrow ? zr_logits_narrow(ctx, V, mb, H, d.A[0], d.lda[0], d_h, H, d_logits, V, d_b_d, (float*)scratch, stream)
                : zr_logits_split(ctx, V, mb, H, d.A[0], d.lda[0], d_h, H, d_logits, V, d_b_d, (float*)scratch, stream, plan.tn, plan.waves);
    if (rc) return rc;
    *partials_out = (float*)scratch;
    *nblocks_out = nblocks;
    return ZR_OK;
  }
  d.B[0] = d_h;
  d.ldb[0] = H;
  const bool split = mb > 256 && zr_split_gemm_takes_product(V, mb, H, false, true, ctx->cu_count);
  if (d_h_packed && d.a_pack == 1 && H % 8 == 0 && (((uintptr_t)d_h_packed & 15u) == 0) && !split) {
    d.B[0] = d_h_packed;
    d.b_packed = 1;
  }
  if (d_h_hi && d.a_pack == 2) {  // the producer of h has left its bf16 terms (the GEMM takes them when they suffice)
    d.Bhi[0] = d_h_hi;
    d.Blo[0] = d_h_lo;
  }
  d.C = d_logits;
  d.ldc = V;
  d.batch = 1;
  d.bias = d_b_d;
  d.epilogue = ZR_EPI_SOFTMAX_PARTIAL;
  d.stream_a = stream ? 1 : 0;
  d.partials = (float*)scratch;
  rc = zr_gemm_launch(ctx, d);
  if (rc) return rc;
  *partials_out = (float*)scratch;
  *nblocks_out = nblocks;
  return ZR_OK;
}

inline void* stats_ptr(float* partials, int nblocks, int mb) {
  size_t off = sizeof(float) * 2 * (size_t)nblocks * mb;
  off = (off + 63) & ~(size_t)63;
  return (char*)partials + off;
}

int check_softmax_args(const char* who, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb) {
  ZR_CHECK_ARG(V > 0 && H > 0 && mb > 0, "%s: V = %d, H = %d, mb = %d", who, V, H, mb);
  ZR_CHECK_ARG(mb <= 65535, "%s: mb = %d exceeds 65535", who, mb);
  ZR_CHECK_ARG(d_D && d_b_d && d_h, "%s: null pointer", who);
  return ZR_OK;
}

}  // namespace

extern "C" {

static int softmax_prepare(zr_ctx* ctx, const char* who, const float* d_D, int V, int H, bool bf16) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(d_D != nullptr && V > 0 && H > 0, "%s: d_D null or V = %d, H = %d", who, V, H);
  ZR_CHECK_ARG(!bf16 || H % 16 == 0, "%s: H = %d is not a multiple of 16", who, H);
  const int ldp = (V + 31) / 32 * 32, kp = bf16 ? H : (H + 7) / 8 * 8;
  ZR_CHECK_ARG(8LL * ldp + 8LL * V < (1LL << 31), "%s: V = %d too large", who, V);
  const size_t bytes = (bf16 ? sizeof(unsigned short) : sizeof(float)) * (size_t)kp * ldp;
  int slot = -1;
  for (int i = 0; i < ZR_MAX_PACKED_D; ++i)
    if (ctx->packed_d[i].key == d_D) slot = i;
  if (slot >= 0 && (ctx->packed_d[slot].V != V || ctx->packed_d[slot].H != H ||
                    ctx->packed_d[slot].bf16 != (bf16 ? 1 : 0))) {
    rc = zr_softmax_release(ctx, d_D);
    if (rc) return rc;
    slot = -1;
  }
  if (slot < 0) {
    for (int i = 0; i < ZR_MAX_PACKED_D && slot < 0; ++i)
      if (!ctx->packed_d[i].key) slot = i;
    ZR_CHECK_ARG(slot >= 0, "%s: all %d slots are in use (zr_softmax_release one)", who, ZR_MAX_PACKED_D);
    void* p = zr_dev_alloc(ctx, bytes);
    if (!p) return zr_set_error(ZR_ENOMEM, "%s: allocation of %zu bytes failed", who, bytes);
    ctx->packed_d[slot].d_pack = p;
    ctx->packed_d[slot].V = V;
    ctx->packed_d[slot].H = H;
    ctx->packed_d[slot].ldp = ldp;
    ctx->packed_d[slot].bf16 = bf16 ? 1 : 0;
  }
  rc = bf16 ? zr_pack8_bf16_launch(ctx, d_D, V, H, V, ldp, kp, (unsigned short*)ctx->packed_d[slot].d_pack)
            : zr_pack4_launch(ctx, d_D, V, H, V, ldp, kp, (float*)ctx->packed_d[slot].d_pack);
  if (rc) {
    (void)zr_dev_release(ctx->packed_d[slot].d_pack);
    ctx->packed_d[slot] = zr_ctx::PackedD{};
    return rc;
  }
  ctx->packed_d[slot].key = d_D;
  return ZR_OK;
}

int zr_softmax_prepare(zr_ctx* ctx, const float* d_D, int V, int H) {
  return softmax_prepare(ctx, "zr_softmax_prepare", d_D, V, H, false);
}

int zr_softmax_prepare_bf16(zr_ctx* ctx, const float* d_D, int V, int H) {
  return softmax_prepare(ctx, "zr_softmax_prepare_bf16", d_D, V, H, true);
}

int zr_softmax_release(zr_ctx* ctx, const float* d_D) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  for (int i = 0; i < ZR_MAX_PACKED_D; ++i) {
    if (ctx->packed_d[i].key == d_D && d_D) {
      ZR_HIP(hipStreamSynchronize(ctx->stream));
      (void)zr_dev_release(ctx->packed_d[i].d_pack);
      ctx->packed_d[i] = zr_ctx::PackedD{};
    }
  }
  return ZR_OK;
}

int zr_softmax_forward(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb,
                       int mode, float* d_out, float* d_logits_scratch) {
  return zr_softmax_forward_packed(ctx, d_D, d_b_d, V, H, d_h, nullptr, mb, mode, d_out, d_logits_scratch);
}

int zr_softmax_block_count(int V) { return V > 0 ? zr_softmax_partial_blocks(V) : 0; }

long long zr_softmax_blocks_offset(int V, int cols) {
  return (V > 0 && cols > 0) ? (long long)zr_softmax_blocks_offset_floats(V, cols) : 0;
}

}  // extern "C"

int zr_softmax_colstats_launch(zr_ctx* ctx, const float* d_partials, int nblocks, int cols, float* d_colstats) {
  softmax_colstats_kernel<<<cols, 256, 0, ctx->stream>>>(d_partials, nblocks, d_colstats);
  ZR_LAUNCH_CHECK("softmax_colstats_kernel");
  return ZR_OK;
}

int zr_softmax_forward_packed(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h,
                              const float* d_h_packed, int mb, int mode, float* d_out, float* d_logits_scratch,
                              const unsigned short* d_h_hi, const unsigned short* d_h_lo) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  rc = check_softmax_args("zr_softmax_forward", d_D, d_b_d, V, H, d_h, mb);
  if (rc) return rc;
  ZR_CHECK_ARG(d_out != nullptr, "zr_softmax_forward: d_out is null");
  ZR_CHECK_ARG(mode == ZR_SOFTMAX_PROB || mode == ZR_SOFTMAX_LOGPROB || mode == ZR_SOFTMAX_LOGITS ||
                   mode == ZR_SOFTMAX_LOGITS_BLOCKS,
               "zr_softmax_forward: mode = %d", mode);
  const bool with_blocks = mode == ZR_SOFTMAX_LOGITS_BLOCKS;
  const bool logits_only = mode == ZR_SOFTMAX_LOGITS || with_blocks;
  ZR_CHECK_ARG(!logits_only || d_logits_scratch == nullptr,
               "zr_softmax_forward: ZR_SOFTMAX_LOGITS(_BLOCKS) writes the logits to d_out and takes no d_logits_scratch");
  float* logits = (d_logits_scratch && !logits_only) ? d_logits_scratch : d_out;
  float* partials = nullptr;
  int nblocks = 0;
  // ZR_SOFTMAX_LOGITS_BLOCKS: the product's per-block pairs go straight into the caller's buffer behind the logits and
  // that is all -- no launch folds them; the consumer (zr_beam_expand_blocks) does that itself
  rc = logits_with_partials(ctx, d_D, d_b_d, V, H, d_h, mb, logits, &partials, &nblocks, d_h_packed, d_h_hi, d_h_lo,
                            with_blocks ? d_out + zr_softmax_blocks_offset_floats(V, mb) : nullptr);
  if (rc) return rc;
  if (with_blocks) return ZR_OK;
  if (logits_only) {
    // ZR_SOFTMAX_LOGITS: the column statistics go behind the logits in the caller's buffer and no normalised matrix is
    // written -- a consumer that needs only a few entries per column (the beam search) normalises those itself
    return zr_softmax_colstats_launch(ctx, partials, nblocks, mb, d_out + (size_t)V * mb);
  }
  float* colstats = (float*)stats_ptr(partials, nblocks, mb);
  return mode == ZR_SOFTMAX_PROB ? launch_normalize<0>(ctx, logits, d_out, V, mb, partials, nblocks, colstats)
                                 : launch_normalize<1>(ctx, logits, d_out, V, mb, partials, nblocks, colstats);
}

int zr_softmax_error_chunks(int V, int n) { return (n + zr_softmax_error_cols(V, n) - 1) / zr_softmax_error_cols(V, n); }

int zr_softmax_error(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int n,
                     const int* d_target, const int* d_mask01, float* d_out, size_t bytes, void** out) {
  float* partials = nullptr;
  int nblocks = 0;
  int rc = logits_with_partials(ctx, d_D, d_b_d, V, H, d_h, n, d_out, &partials, &nblocks);
  if (rc) return rc;
  float* colstats = (float*)stats_ptr(partials, nblocks, n);
  softmax_colstats_kernel<<<n, 256, 0, ctx->stream>>>(partials, nblocks, colstats);
  ZR_LAUNCH_CHECK("softmax_colstats_kernel");
  rc = zr_ctx_scratch(ctx, 0, bytes, out);
  if (rc) return rc;
  float* sums = (float*)*out;
  const int chunks = zr_softmax_error_chunks(V, n), cols = zr_softmax_error_cols(V, n);
  float* p_target = sums + (((size_t)V * chunks + 3) & ~(size_t)3);
  if (V % 4 == 0 && (((uintptr_t)d_out & 15u) == 0)) {
    const dim3 grid((V / 4 + 255) / 256, chunks);
    softmax_error_kernel<true><<<grid, 256, 0, ctx->stream>>>(d_out, V, n, cols, colstats, d_target, d_mask01, sums, p_target);
  } else {
    const dim3 grid((V + 255) / 256, chunks);
    softmax_error_kernel<false><<<grid, 256, 0, ctx->stream>>>(d_out, V, n, cols, colstats, d_target, d_mask01, sums, p_target);
  }
  ZR_LAUNCH_CHECK("softmax_error_kernel");
  return ZR_OK;
}

extern "C" {

// zr_softmax_forward on the device's statically allocated scratch array: same kernels, no allocation.  The array is
// split into the two buffers the product needs (re-laid-out activations, then partial column statistics + column
// statistics); both are fully written before they are read, so nothing has to be cleared between calls.
int zr_softmax_forward_static(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb,
                              int mode, float* d_out, float* d_logits_scratch) {
  ZR_CHECK_ARG(ctx != nullptr && ctx->d_static_scratch != nullptr, "zr_softmax_forward_static: null context");
  ctx->fixed_scratch = 1;
  ctx->d_fixed[0] = ctx->d_static_scratch;
  ctx->fixed_bytes[0] = ZR_STATIC_SCRATCH_SLOT0_BYTES;
  ctx->d_fixed[1] = (char*)ctx->d_static_scratch + ZR_STATIC_SCRATCH_SLOT0_BYTES;
  ctx->fixed_bytes[1] = ZR_STATIC_SCRATCH_BYTES - ZR_STATIC_SCRATCH_SLOT0_BYTES;
  const int rc = zr_softmax_forward(ctx, d_D, d_b_d, V, H, d_h, mb, mode, d_out, d_logits_scratch);
  ctx->fixed_scratch = 0;
  return rc;
}

int zr_softmax_logprob_f64(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb,
                           double* d_logp, float* d_logits_scratch) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  rc = check_softmax_args("zr_softmax_logprob_f64", d_D, d_b_d, V, H, d_h, mb);
  if (rc) return rc;
  ZR_CHECK_ARG(d_logp && d_logits_scratch, "zr_softmax_logprob_f64: null output or scratch");
  float* partials = nullptr;
  int nblocks = 0;
  rc = logits_with_partials(ctx, d_D, d_b_d, V, H, d_h, mb, d_logits_scratch, &partials, &nblocks);
  if (rc) return rc;
  double* colstats = (double*)stats_ptr(partials, nblocks, mb);
  softmax_colstats_f64_kernel<<<mb, kF64Threads, 0, ctx->stream>>>(d_logits_scratch, V, partials, nblocks, colstats, nullptr);
  ZR_LAUNCH_CHECK("softmax_colstats_f64_kernel");
  dim3 grid((V + 255) / 256, mb);
  softmax_logprob_f64_kernel<<<grid, 256, 0, ctx->stream>>>(d_logits_scratch, d_logp, V, colstats);
  ZR_LAUNCH_CHECK("softmax_logprob_f64_kernel");
  return ZR_OK;
}

int zr_softmax_loss(zr_ctx* ctx, const float* d_D, const float* d_b_d, int V, int H, const float* d_h, int mb,
                    const int* d_target, const int* d_mask01, float* d_logits_scratch, double* h_loss) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  rc = check_softmax_args("zr_softmax_loss", d_D, d_b_d, V, H, d_h, mb);
  if (rc) return rc;
  ZR_CHECK_ARG(d_target && d_mask01 && d_logits_scratch && h_loss, "zr_softmax_loss: null pointer");
  float* partials = nullptr;
  int nblocks = 0;
  rc = logits_with_partials(ctx, d_D, d_b_d, V, H, d_h, mb, d_logits_scratch, &partials, &nblocks);
  if (rc) return rc;
  double* colstats = (double*)stats_ptr(partials, nblocks, mb);
  // enough workgroups for two a compute unit, each with at least one round of loads
  int parts = (2 * ctx->cu_count + mb - 1) / mb;
  const int rounds = V / (4 * kF64Threads * 4);
  parts = parts < rounds ? parts : rounds;
  parts = parts > 16 ? 16 : (parts < 1 ? 1 : parts);
  void* sums = nullptr;
  if (parts > 1) {  // (the product is done with this buffer)
    if (zr_ctx_scratch(ctx, 0, sizeof(double) * (size_t)parts * mb, &sums) != ZR_OK) parts = 1;
  }
  softmax_colstats_f64_kernel<<<dim3(mb, parts), kF64Threads, 0, ctx->stream>>>(d_logits_scratch, V, partials, nblocks, colstats, (double*)sums);
  ZR_LAUNCH_CHECK("softmax_colstats_f64_kernel");
  // the loss cell lives in the partials area, which is dead once the column stats exist
  double* d_loss = (double*)partials;
  softmax_loss_kernel<<<1, 256, 0, ctx->stream>>>(d_logits_scratch, V, mb, colstats, (const double*)sums, parts, d_target, d_mask01, d_loss,
                                                  ctx->d_flags);
  ZR_LAUNCH_CHECK("softmax_loss_kernel");
  ZR_HIP(hipMemcpyAsync(h_loss, d_loss, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  ZR_HIP(hipStreamSynchronize(ctx->stream));
  return ZR_OK;
}

}  // extern "C"
