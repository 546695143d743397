// Whole-sweep kernel with streamed weights: ONE launch runs every (layer, time step) node of a stacked forward pass, its products on
// the bf16 matrix cores with every fp32 operand as three exact bf16 terms (zr_split_gemm.hip says why that loses nothing).
//
// A workgroup owns the same tile -- 32 hidden rows x 32*TN batch columns of one layer -- at every time step and loops
// over t itself.  Node (l, t) needs h of (l-1, t) and of (l, t-1), each produced by the j_tiles workgroups that own
// the same batch columns of that layer: every (layer, column tile) has an arrival counter in device memory that its
// producers bump once per time step, and a consumer waits until the counter reaches (steps needed) * j_tiles.
// Compared with one launch per diagonal this removes, per step, the launch, the drain of the slowest tile and the
// refill of the operand pipeline from a cold start; the cell state never leaves registers.
//
// Eight waves: wave w has gate w % 4 and, of every 64 k, the first or second 32 (w / 4).  Its weights come from memory straight
// into its registers, four steps of 64 k ahead and on into the next time step, and are split there: no other wave of the
// workgroup needs them.  The activations' terms go through LDS: h is handed from node to node already split, 16-byte items of 8 k of one
// term; embedding columns and h0 are split on their way in.  The two waves on a SIMD split and multiply in turn.  Twelve products of 32 k
// are summed from zero before they reach the accumulator (short chains, one rounding at its size).
// A loop over steps has no branch: waits for producers come before it or at the start of four steps, what lies past the end is
// loaded as zero.  (With branches around loads the compiler waits for all of them at once: the sweep named next took 3100 us.)
//
// Bound by the matrix cores' rate under load and the hand-overs: 4 layers of H = 1000, 128 columns, 50 steps 3250 us on the fp32 matrix instructions,
// 2490 to 2710 here by the run, 2600 on average: 409.6 GFLOP = 158 TFLOP/s, 0.95 PFLOP/s of bf16 work where large bf16 products reach 1.2 on this card; a
// steady step 49 to 52 us.  64 columns of it, 20 steps, 770 -> 705 (32-column tiles, whose weights are split for half the products).  Error of h against 64 bits, here and
// with the fp32 instructions: H = 64 1.5e-7 / 1.6e-7, 512 1.9e-7 / 2.3e-7, 1000 2.1e-7 / 5.1e-7.
//
// Hand-over through memory: h is written twice, to the caller's array (plain stores, visible at kernel end) and as three terms
// [term][H/8][mb][8] per (layer, t) that the consumers read.  The chip's eight dies have one L2 each.
// The terms are written with device-scope stores (written through to memory); every wave waits for its stores to
// complete, then a workgroup barrier, then one thread bumps the counter.  A consumer polls the counter with
// device-scope loads and reads the terms with ordinary loads.  Those cannot hit a stale line as long as no line is
// cached before it was written: caches are clean when the kernel starts, every line is read only after
// the wait for its producers, and with the columns padded to a multiple of eight a 128-byte line (8 columns of 8 rows) has one producer.
// (Invalidating the caches after every wait instead throws out the weights: 4 layers of H = 1000, 100 columns, 12 steps 908 us.)
//
// Progress: the launch must be wholly resident (the host checks grid <= CUs x resident workgroups per CU), then the
// dependency graph is acyclic and every wait ends.  Every wait is bounded all the same: a workgroup that runs out of
// polls marks every counter, which releases all other waiters, raises the status flag and leaves; the others leave
// at their next wait.
#include "zr_internal.h"
#include "zr_lstm_sweep.h"
#include "zr_math.h"
#include "zr_mfma_core.h"

namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any multiple of 4
typedef unsigned zr_u32x2 __attribute__((ext_vector_type(2)));

// All threads of the workgroup call this.  False: leave the kernel.
__device__ __forceinline__ bool sweep_wait(const LstmSweep& P, int* ctr, int target, int* s_go) {
  if (threadIdx.x == 0) {
    int v = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int spins = 0; v < target && spins < P.spin_limit; ++spins) {
      __builtin_amdgcn_s_sleep(8);
      v = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool ok = v >= target && !(v & kSweepGaveUp);
    if (!ok) {
      if (!(v & kSweepGaveUp)) {
        const int n = P.nl * P.n_tiles;
        for (int i = 0; i < n; ++i) atomicOr(P.counters + i * kSweepCtrStride, kSweepGaveUp);
      }
      __hip_atomic_store(P.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    *s_go = ok ? 1 : 0;
  }
  __syncthreads();
  return *s_go != 0;
}

// The embedding columns of every time step and the initial states as terms.  Eight lanes take 64 k of a column, so that reads and writes are
// whole lines; blockIdx.z: the embedding (T * mb columns), then each layer's h0 (mb columns).
__global__ void __launch_bounds__(256) lstm_sweep_terms_kernel(LstmSweep P) {
  const int kg = blockIdx.y * 8 + (threadIdx.x & 7), H = P.H, mb = P.mb;
  const int which = blockIdx.z, c = blockIdx.x * 32 + (threadIdx.x >> 3);
  if (8 * kg >= H || c >= (which ? mb : P.T * mb)) return;
  const long long n_el = (long long)H * P.columns, slot = 3 * n_el;
  const int t = which ? 0 : c / mb, n = c - t * mb;
  const float* x = which ? P.h0[which - 1] + (long long)n * H : P.embed + (long long)P.clamp_id(P.ids[c]) * H;
  unsigned short* d = (which ? P.hp + (long long)(which - 1) * (P.T + 1) * slot : P.xp + t * slot) + ((long long)kg * P.columns + n) * 8;
  zr_u32x4 term[3];
  const zr_f32x4 lo = *(const f32x4u*)(x + 8 * kg), hi = *(const f32x4u*)(x + 8 * kg + 4);
  zr_split_terms(lo, hi, term);
#pragma unroll
  for (int q = 0; q < 3; ++q) *(zr_u32x4*)(d + q * n_el) = term[q];
}

template <int TN>
__global__ void __launch_bounds__(512, 2) lstm_sweep_kernel(LstmSweep P) {
  constexpr int COLS = 32 * TN, TERM = 8 * COLS, BUF = 3 * TERM;  // 16-byte items: of one term's 64 k, of all terms
  constexpr int RING = 4;                  // steps of 64 k that the weights are ahead
  constexpr int ROWS = 2 * TN;             // hidden rows of a thread in the cell update: 16 / TN threads a column
  constexpr int ZP = 36;                   // floats of a column's 32 rows in `zs`, padded off the banks of the next column
  constexpr bool ALL = 8 * COLS == 512;    // every thread fetches activations
  __shared__ zr_u32x4 s[2 * BUF];
  __shared__ __align__(16) float zs[2 * 4 * COLS * ZP];
  __shared__ int s_go[2];
  // Workgroup ids congruent modulo 8 share a die: the column tiles of a row tile are neighbours on one die and read its weights together.
  const int r8 = blockIdx.x & 7;
  const int q8 = blockIdx.x >> 3;
  const int nt = q8 % P.n_tiles;
  const int groups = P.nl * P.j_tiles;
  const int group = r8 * ((groups + 7) >> 3) + q8 / P.n_tiles;
  if (q8 / P.n_tiles >= ((groups + 7) >> 3) || group >= groups) return;
  const int l = group / P.j_tiles;
  const int jt = group % P.j_tiles;

  const int tid = threadIdx.x, lane = tid & 63, jl = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gate = wave & 3, kh = wave >> 2;
  const int H = P.H, mb = P.mb;
  const int j0 = jt * 32, n0 = nt * COLS;
  const long long n_el = (long long)H * P.columns;  // of a term of a state
  const int nit = (H + 127) >> 7 << 1, steps = 2 * nit;  // steps of 64 k: of a segment, of a node (a multiple of RING)

  // Weights: element (row, k) of matrix m at ((k/4)*ldw + row)*4 + k%4; a descriptor that ends with the matrix reads zeros past kp.
  const long long HH = (long long)P.kp * P.ldw;
  const unsigned kblock = 16u * (unsigned)P.ldw;  // bytes of four k
  const unsigned woff = 16u * (unsigned)(j0 + jl) + (unsigned)(8 * kh + 2 * half) * kblock;
  zr_f32x4 ar[RING][4];
  // Segment 0: the input from below, 1: h of (l, t-1).  Layers above the first take the recurrent segment first: it only needs the layer's own
  // previous step, so a layer can trail the one below it by half a step instead of a whole one (the pipeline of layers fills and
  // drains in half the time: 2 % of a sweep of 4 layers of H = 1000, 128 columns, 50 steps) and the wait for the layer below hides behind half a K loop.
  // The order is fixed per layer, so that no bit of the result depends on timing.
  auto seg_of = [&](int v) { return (v >= nit) != (l > 0) ? 1 : 0; };
  auto load_a = [&](zr_f32x4 (&a)[4], int v) {
    const int it = v >= nit ? v - nit : v;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(P.W[l] + (seg_of(v) * 4 + gate) * HH), 0,
                                                                       (int)(unsigned)(HH * 4), 0x00020000);
#pragma unroll
    for (int i = 0; i < 4; ++i)  // blocks of four k: 0, 1, 4, 5 (half 0), 2, 3, 6, 7 (half 1)
      a[i] = __builtin_bit_cast(zr_f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              r, (int)(woff + (unsigned)(16 * it + (i & 1) + 4 * (i >> 1)) * kblock), 0, 0));
  };

  // This thread's item of the activations of a step: eight k of one column.
  const int bkg = tid / COLS, bcol = n0 + tid % COLS < mb ? n0 + tid % COLS : mb - 1;
  const bool fetches = ALL || tid < 8 * COLS;  // uniform over a wave
  // This thread's outputs: rows cr .. cr + ROWS - 1 of column cn.
  const int cr = ROWS * (tid & (16 / TN - 1)), cn = tid / (16 / TN);
  const int j = j0 + cr, n = n0 + cn;
  const bool out_ok = j < H && n < mb;  // H is a multiple of 8
  const int jc = j < H ? j : 0, nc = n < mb ? n : mb - 1;

  float c_state[ROWS];
#pragma unroll
  for (int e = 0; e < ROWS; ++e) c_state[e] = P.c0[l][(long long)nc * H + jc + e];
  int* my_ctr = P.counters + (l * P.n_tiles + nt) * kSweepCtrStride;
  int* below_ctr = P.counters + ((l > 0 ? l - 1 : 0) * P.n_tiles + nt) * kSweepCtrStride;
  // Terms of one state: [3][H/8][columns][8].  Slot t of a layer is its h of time step t - 1, of "layer -1" the embedding columns of step t.
  const long long slot = 3 * n_el;
  unsigned short* hp_mine = P.hp + (long long)l * (P.T + 1) * slot;
  const unsigned short* hp_below = l > 0 ? P.hp + ((long long)(l - 1) * (P.T + 1) + 1) * slot : P.xp;

  zr_bf16x8 x[2][3];  // the weights of 16 k in use, and the next 16 k's, split beside the products of these
  auto split_a = [&](const zr_f32x4& lo, const zr_f32x4& hi, zr_bf16x8 (&x)[3]) {
    zr_u32x4 term[3];
    zr_split_terms(lo, hi, term);
#pragma unroll
    for (int q = 0; q < 3; ++q) x[q] = __builtin_bit_cast(zr_bf16x8, term[q]);
  };
#pragma unroll
  for (int u = 0; u < RING; ++u) load_a(ar[u], u);
  split_a(ar[0][0], ar[0][1], x[0]);

  for (int t = 0; t < P.T; ++t) {
    zr_u32x4 bv[2][3];
    // Activations of step v on their way (past k, or past the last step: zeros).
    auto fetch_b = [&](zr_u32x4 (&d)[3], int v) {
      if (!fetches) return;
      const int k = 64 * (v >= nit ? v - nit : v) + 8 * bkg;
      const unsigned short* x = (seg_of(v) == 0 ? hp_below : hp_mine) + (long long)t * slot;
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(x), 0, (int)(unsigned)(6 * n_el), 0x00020000);
      const int off = k < H && v < steps ? (int)(16u * (unsigned)((k >> 3) * P.columns + bcol)) : -16;
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q] = __builtin_bit_cast(zr_u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, (int)(unsigned)(2 * q * n_el), 0));
    };
    auto store_b = [&](const zr_u32x4 (&v)[3], int buf) {
      if (!fetches) return;
      zr_u32x4* d = s + buf * BUF + tid;
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q * TERM] = v[q];
    };
    // The producers of segment q have finished.  False: leave the kernel.
    auto wait_for = [&](int q) {
      const int sg = seg_of(q * nit);
      if (sg == 0 ? l == 0 : t == 0) return true;
      return sweep_wait(P, sg == 0 ? below_ctr : my_ctr, (sg == 0 ? t + 1 : t) * P.j_tiles, &s_go[sg]);
    };

    zr_f32x16 acc[TN];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    auto compute = [&](const zr_f32x4 (&a)[4], const zr_f32x4 (&next)[4], int buf) {
      zr_f32x16 sum[TN] = {};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        zr_bf16x8 y[TN][3];
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          const zr_u32x4* b = s + buf * BUF + (4 * kh + 2 * st + half) * COLS + 32 * i + jl;
#pragma unroll
          for (int q = 0; q < 3; ++q) y[i][q] = __builtin_bit_cast(zr_bf16x8, b[q * TERM]);
        }
        constexpr int X[6] = {2, 0, 1, 1, 0, 0}, Y[6] = {0, 2, 1, 0, 1, 0};  // the smallest products first
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (int i = 0; i < TN; ++i) sum[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[st][X[p]], y[i][Y[p]], sum[i], 0, 0, 0);
        if (st == 0)
          split_a(a[2], a[3], x[1]);
        else
          split_a(next[0], next[1], x[0]);
        // matrix instructions and the conversions in turn (left to the compiler: 8 % slower)
#pragma unroll
        for (int i = 0; i < 6 * TN; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, TN == 2 ? 4 : 8, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < TN; ++i) acc[i] += sum[i];
    };

    if (!wait_for(0)) return;
    fetch_b(bv[0], 0);
    fetch_b(bv[1], 1);
    if (nit == 2 && !wait_for(1)) return;
    store_b(bv[0], 0);
    fetch_b(bv[0], 2);
    __syncthreads();
    for (int c0 = 0; c0 < steps; c0 += RING) {
      // activations are fetched three steps ahead
      if (nit >= c0 + 3 && nit < c0 + 3 + RING && !wait_for(1)) return;
#pragma unroll
      for (int u = 0; u < RING; ++u) {
        const int c = c0 + u;
        // the other buffer was last read in step c - 1, behind the barrier that ended it
        store_b(bv[(u + 1) & 1], (u + 1) & 1);
        // (loads arrive in order: activations, needed first, go out before weights needed later)
        fetch_b(bv[(u + 1) & 1], c + 3);
        compute(ar[u], ar[(u + 1) % RING], u & 1);
        load_a(ar[u], c + RING < steps ? c + RING : c + RING - steps);
        __syncthreads();
      }
    }

    // Terms of an infinite operand are infinity and NaN: sums that come out infinite or NaN are computed again with fp32
    // instructions, from the operands themselves (h, which is bounded, as the exact sum of its terms).
    bool finite = true;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) finite = finite && fabsf(acc[i][r]) <= 3.402823466e38f;
    if (__any(!finite)) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
      for (int sg = 0; sg < 2; ++sg) {
        const float* W = P.W[l] + (sg * 4 + gate) * HH;
        const bool terms = sg == 0 ? l > 0 : t > 0;
        const unsigned short* x = (sg == 0 ? hp_below : hp_mine) + (long long)t * slot;
        for (int k = 32 * kh; k < H; k = (k & 31) == 30 ? k + 34 : k + 2) {  // H is even
          const int kk = k + half;
          const float w = W[((long long)(kk >> 2) * P.ldw + j0 + jl) * 4 + (kk & 3)];
#pragma unroll
          for (int i = 0; i < TN; ++i) {
            const int col = n0 + 32 * i + jl < mb ? n0 + 32 * i + jl : mb - 1;
            float v;
            if (terms) {
              const unsigned short* b = x + ((long long)(kk >> 3) * P.columns + col) * 8 + (kk & 7);
              v = __uint_as_float((unsigned)b[0] << 16) + (__uint_as_float((unsigned)b[n_el] << 16) + __uint_as_float((unsigned)b[2 * n_el] << 16));
            } else if (sg == 0) {
              v = P.embed[(long long)P.clamp_id(P.ids[(long long)t * mb + col]) * H + kk];
            } else {
              v = P.h0[l][(long long)col * H + kk];
            }
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(w, v, acc[i], 0, 0, 0);
          }
        }
      }
    }

    // A lane has one column of each 32 x 32 block and sixteen of its rows.
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(zr_f32x4*)(zs + ((kh * 4 + gate) * COLS + 32 * i + jl) * ZP + 8 * q + 4 * half) =
            zr_f32x4{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
    const float mask = (float)P.mask01[(long long)t * mb + nc];
    float bias[4][ROWS];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < ROWS; ++e) bias[g][e] = P.bias[l][g * H + jc + e];
    __syncthreads();
    float z[4][ROWS], h_v[ROWS], g_v[4][ROWS];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < ROWS; ++e)
        z[g][e] = zs[(g * COLS + cn) * ZP + cr + e] + zs[((4 + g) * COLS + cn) * ZP + cr + e] + bias[g][e];
#pragma unroll
    for (int e = 0; e < ROWS; ++e) {
      float c;
      zr_lstm_cell(z[0][e], z[1][e], z[2][e], z[3][e], c_state[e], mask, P.clip, g_v[0][e], g_v[1][e], g_v[2][e], g_v[3][e], c, h_v[e]);
      c_state[e] = c;
    }
    // Only the terms of h, which the waiting workgroups read, go out before the arrival is published;
    // the outputs nobody waits for (h, c and the gate values kept for training) are stored after it.
    if (out_ok) {
      unsigned short* d = hp_mine + (long long)(t + 1) * slot + ((long long)(j >> 3) * P.columns + n) * 8 + (j & 7);
      float left[ROWS];
#pragma unroll
      for (int e = 0; e < ROWS; ++e) left[e] = h_v[e];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        if constexpr (TN == 2) {
          const unsigned lo = zr_next_terms(left[0], left[1]), hi = zr_next_terms(left[2], left[3]);
          __hip_atomic_store((unsigned long long*)(d + q * n_el), lo | (unsigned long long)hi << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          __hip_atomic_store((unsigned*)(d + q * n_el), zr_next_terms(left[0], left[1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    // publish this step: every wave's stores have completed before the barrier, then one arrival per workgroup
    zr_publish_barrier();
    if (tid == 0) atomicAdd(my_ctr, 1);
    if (out_ok) {
      const long long state = (long long)H * mb, ix = t * state + (long long)n * H + j;
      float* gates = P.gates_all[l];
#pragma unroll
      for (int e = 0; e < ROWS; ++e) {
        P.c_all[l][ix + e] = c_state[e];
        P.h_all[l][ix + e] = h_v[e];
      }
      if (gates) {
        float* gt = gates + 3 * t * state + ix;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < ROWS; ++e) gt[g * state + e] = g_v[g][e];
      }
    }
  }
}

}  // namespace

int zr_sweep_capacity(zr_ctx* ctx, int tn) {
  int& cached = ctx->sweep_capacity[tn];
  if (cached == 0) {
    int cus = 0, per_cu = 0;
    const void* kernel = tn == 1 ? (const void*)lstm_sweep_kernel<1> : (const void*)lstm_sweep_kernel<2>;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 512, 0) != hipSuccess) {
      (void)hipGetLastError();
      cached = -1;
    } else {
      ctx->cu_count = cus;
      cached = cus * per_cu > 0 ? cus * per_cu : -1;
    }
  }
  return cached > 0 ? cached : 0;
}

int zr_sweep_launch(zr_ctx* ctx, const LstmSweep& P, int tn) {
  const int grid = (P.nl * P.j_tiles + 7) / 8 * 8 * P.n_tiles;
  lstm_sweep_terms_kernel<<<dim3(((long long)P.T * P.mb + 31) / 32, (P.H + 63) / 64, 1 + P.nl), 256, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("lstm_sweep_terms_kernel");
  if (tn == 1)
    lstm_sweep_kernel<1><<<grid, 512, 0, ctx->stream>>>(P);
  else
    lstm_sweep_kernel<2><<<grid, 512, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("lstm_sweep_kernel");
  return ZR_OK;
}
