// The backward sweep of a stack with the weights held in registers: all time steps of as many layers as fit the device in one launch,
// for small models and narrow batches (H up to 512, any H from 8).
//
// One launch per anti-diagonal for the gate derivatives and one for the error products is two launches and two trips through memory for a few
// microseconds' work: 12.4 us a diagonal at 2 x 300, 20 columns.  As in lstm_resident_kernel (zr_lstm_resident.hip) a workgroup
// keeps its weights for all steps: 16 hidden rows of one layer, for which it owes the errors.  They are sums over the four gate errors of all rows,
// Wh^T of its own layer (error to h_{t-1}) and M^T of the layer above: 16 x 8H floats over 512 threads, H/4 registers each.  Then the
// cell's derivatives of its own rows run in registers, the cell error never leaves them, and only the gate errors travel, [row][column][gate], a
// k-group of the products being four rows' four gates.  The last role has the rows of M^T of layer 0 and makes the error to the input from below, in a
// launch of its own where there is no room for it beside the layers.
// Bound: the chain of time steps -- gate errors of (l, t+1) published by every row tile, seen, multiplied, before those of (l, t) --
// which the product with the layer above, there a step early, is kept off, and so are the cell's derivatives: 2.7 us a step at H = 64,
// 5.7 at 300, 8.9 at 500 (of which 3.7 are matrix instructions, half-rate for want of columns).  Whole sweeps, us, per diagonal / so: 1 x 64, 8 columns,
// 40 steps 320 / 112; 2 x 300, 20 columns, 35 steps 421 / 210; 2 x 500, 64 columns, 24 steps 405 / 230.
//
// Hand-over, waits and their bound as in the forward kernel: device-scope stores, one flag per workgroup, columns padded to eight so
// that a 128-byte line has one producer, and read only behind its flag.  A workgroup that gives up a wait marks its flag and the launch; then
// lstm_backward_redo_kernel, which is always queued behind it and otherwise leaves at once, forms everything again, one workgroup a
// column and no waits between workgroups.  So the call cannot fail where the launches per diagonal did not.
#include "zr_internal.h"
#include "zr_mfma_core.h"

namespace {

constexpr int kMaxLayers = 16;
constexpr int kWaves = 8;              // waves per workgroup = K slices
constexpr int kRows = 16;              // hidden rows a workgroup
constexpr int kCols = 16;              // columns a workgroup
constexpr int kRedLd = 20;             // LDS row of 16 partial sums, padded
constexpr int kRedSeg = kCols * kRedLd + 32;
constexpr int kGaveUp = 1 << 28;

struct BackResident {
  const float* stack[kMaxLayers];  // [2][H x 4H]: element (k, g*H + j) = W_g[j][k] at k + (g*H + j)*H, of Wh and of M
  const float* gates[kMaxLayers];
  const float* c[kMaxLayers];
  const float* c0[kMaxLayers];
  const float* err_hT[kMaxLayers];  // null: zero
  const float* err_cT[kMaxLayers];
  float* dgates[kMaxLayers];
  float* err_h0[kMaxLayers];
  float* err_c0[kMaxLayers];
  const float* err_top;
  float* err_below0;              // null: not wanted here
  const int* mask01;
  float* dp;                      // [nl][T] slots of [16 j_tiles][mbp][4]: the gate errors of (l, t) in slot T - 1 - t
  long long slot;
  int* flags;                     // [layers of this launch][n_tiles][flag_stride], zero at launch: slots published
  int flag_stride, n_flags;
  int* departures;
  int* failed;                    // set to `epoch` when a wait was abandoned
  int epoch;
  int l_top, layers, below_parts;  // this launch: layers l_top, l_top - 1, ..., and workgroups that share the steps of the error to the input from below
  int nl, T, H, mb, mbp, j_tiles, n_tiles;
  float clip;
  int spin_limit;
  int wait_extra;                 // 0; in tests of giving up waits want so many slots more than there are
};

__device__ __forceinline__ float clamp_error(float v, float clip) { return v > clip ? clip : (v < -clip ? -clip : v); }

// A point of lstm_node_backward_group_kernel (zr_backward.hip): what does not depend on the errors ...
struct Slopes {
  float c, d[4], f;  // of the cell error by h's, of the gate errors by the cell's (d[3]: by h's), the forget gate
};
__device__ __forceinline__ Slopes node_slopes(const float (&g)[4], float c, float cprev) {
  const float th = tanhf(c);
  return {g[3] * (1.0f - th * th), {g[2] * g[0] * (1.0f - g[0]), cprev * g[1] * (1.0f - g[1]), g[0] * (1.0f - g[2] * g[2]), th * g[3] * (1.0f - g[3])}, g[1]};
}
// ... and the gate errors and the error to c_{t-1} (in ec) from the error at h.
__device__ __forceinline__ void node_point(float eh, float m, const Slopes& s, float& ec, float (&d)[4]) {
  eh *= m;
  const float e = (ec + eh * s.c) * m;
  d[0] = e * s.d[0];
  d[1] = e * s.d[1];
  d[2] = e * s.d[2];
  d[3] = eh * s.d[3];
  ec = e * s.f;
}

// NG: k-groups (four rows' gate errors) per wave and segment, H <= 32 * NG.
template <int NG>
__global__ void __launch_bounds__(64 * kWaves, NG <= 4 ? 4 : 2) lstm_backward_resident_kernel(BackResident P) {
  __shared__ float red[kWaves * 2 * kRedSeg];
  __shared__ int s_abort, s_last;
  const int tid = threadIdx.x, lane = tid & 63;
  const int kslice = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = P.H, mb = P.mb;
  const size_t n = (size_t)H * mb;
  const int nt = (int)blockIdx.x % P.n_tiles;
  const int jt = ((int)blockIdx.x / P.n_tiles) % P.j_tiles;
  const int role = (int)blockIdx.x / (P.n_tiles * P.j_tiles);
  const bool below = role >= P.layers;  // M^T of layer 0 and nothing else
  const int l = below ? -1 : P.l_top - role;
  const int j0 = jt * kRows, n0 = nt * kCols;
  const int cl = lane & 15, kq = lane >> 4;
  if (tid == 0) s_abort = 0;
  __syncthreads();

  auto work = [&]() {
    const bool top = l == P.nl - 1;
    // ---- weights: w[0] with the layer's own step t + 1, w[1] with the layer above
    float w[2][NG][4];
    const int out = j0 + cl < H ? j0 + cl : H - 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bool have = s == 0 ? !below : !top;
      const float* m = have ? P.stack[s == 0 ? l : l + 1] + (size_t)s * 4 * H * H + out : nullptr;
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const int j = 4 * (kslice + kWaves * i) + kq;
#pragma unroll
        for (int g = 0; g < 4; ++g) w[s][i][g] = have && j < H ? m[((size_t)g * H + j) * H] : 0.0f;
      }
    }
    // ---- the point this thread finishes together with its neighbour: lane pairs share one, each adds up one segment
    const int seg = tid & 1, o = tid >> 1, oj = o & 15, on = o >> 4;
    const int j = j0 + oj, b = n0 + on;
    const bool ok = j < H && b < mb;
    const size_t ix = (size_t)(b < mb ? b : mb - 1) * H + (j < H ? j : H - 1);
    const unsigned dp_at = (unsigned)(((size_t)j * P.mbp + (b < mb ? b : mb - 1)) * 4 + 2 * seg);
    // ---- flags: the producers of a wave's groups are every other row tile
    int* flags_here = below ? nullptr : P.flags + (role * P.n_tiles + nt) * P.flag_stride;
    const int above_role = (below ? P.layers : role) - 1;  // (-1: made by an earlier launch)
    const int* flags_above = above_role >= 0 ? P.flags + (above_role * P.n_tiles + nt) * P.flag_stride : nullptr;
    const int tile = 2 * lane + (kslice >> 2);
    const bool looks = lane < NG && tile < P.j_tiles;
    bool dead = false;
    auto wait_for = [&](const int* flags, int target) {
      if (dead) return;
      target += P.wait_extra;
      int spins = 0;
      bool gave_up = false;
      for (;;) {
        const int v = looks ? __hip_atomic_load(flags + tile, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : kGaveUp - 1;
        if (__all(v >= target)) {
          gave_up = __any(v >= kGaveUp);
          break;
        }
        if (++spins > P.spin_limit) {
          gave_up = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      if (gave_up) {
        dead = true;
        if (lane == 0) s_abort = 1;
      }
      asm volatile("" ::: "memory");  // nothing behind the wait is read before it
    };
    const int col = n0 + cl < mb ? n0 + cl : mb - 1;
    const int n_groups = 4 * P.j_tiles;  // (a line that nobody writes, or that is read before its flag, would go stale)
    const float* dp_here = below ? nullptr : P.dp + (size_t)l * P.T * P.slot;
    const float* dp_above = top ? nullptr : P.dp + (size_t)(l + 1) * P.T * P.slot;
    // Four accumulators, one a gate, while a segment is multiplied: chains a fourth as long.  (With two the errors were up to 13 % farther
    // from 64 bits than the launches per diagonal leave them.)
    zr_f32x4 acc[2];
    auto product = [&](int s, const float* slot) {
      zr_f32x4 a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      constexpr int AHEAD = NG > 12 ? 7 : NG;  // in flight at once: all of a wave's groups where the registers allow it
      zr_f32x4 x[AHEAD];
      auto load = [&](int i) {
        const int g = kslice + kWaves * i;
        x[i % AHEAD] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (g < n_groups) x[i % AHEAD] = *(const zr_f32x4*)(slot + ((unsigned)(4 * g + kq) * (unsigned)P.mbp + (unsigned)col) * 4u);
      };
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) load(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NG; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i % AHEAD][e], w[s][i][e], a[e], 0, 0, 0);
        if (i + AHEAD < NG) {
          load(i + AHEAD);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      acc[s] = (a[0] + a[1]) + (a[2] + a[3]);
    };
    auto clear = [&]() {
      acc[0] = acc[1] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    // This thread's segment's sum over the K slices; false: a wave of this workgroup gave up.  The sums may be written again
    // behind the next barrier.
    auto reduce = [&](float& sum) {
      float* mine = red + kslice * 2 * kRedSeg + 4 * kq * kRedLd + cl;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[s * kRedSeg + r * kRedLd] = acc[s][r];
      __syncthreads();
      if (s_abort) return false;
      const float* p = red + seg * kRedSeg + on * kRedLd + oj;
      float part[kWaves];
#pragma unroll
      for (int q = 0; q < kWaves; ++q) part[q] = p[q * 2 * kRedSeg];
      sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
      return true;
    };
    auto abandon = [&]() {
      if (tid == 0) {
        if (flags_here) __hip_atomic_store(flags_here + jt, kGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(P.failed, P.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    };

    if (below) {
      for (int s = role - P.layers; s < P.T; s += P.below_parts) {
        clear();
        if (flags_above) wait_for(flags_above, s + 1);
        product(1, dp_above + (size_t)s * P.slot);
        float sum;
        if (!reduce(sum)) return abandon();
        if (ok && seg == 1) P.err_below0[(size_t)(P.T - 1 - s) * n + ix] = sum;
        __syncthreads();
      }
      return;
    }

    // what a step needs besides the errors, asked for a step ahead
    float gv[4], c_now, c_before, top_v = 0.0f, mask_v, ec = P.err_cT[l] ? P.err_cT[l][ix] : 0.0f;
    auto fetch = [&](int t) {
      const float* gt = P.gates[l] + (size_t)t * 4 * n + ix;
#pragma unroll
      for (int g = 0; g < 4; ++g) gv[g] = gt[g * n];
      c_before = t ? P.c[l][(size_t)(t - 1) * n + ix] : P.c0[l][ix];
      if (top) top_v = P.err_top[(size_t)t * n + ix];
      mask_v = (float)P.mask01[(size_t)t * mb + (b < mb ? b : mb - 1)];
    };
    c_now = P.c[l][(size_t)(P.T - 1) * n + ix];
    fetch(P.T - 1);
    float next0 = P.err_hT[l] ? P.err_hT[l][ix] : 0.0f;
    for (int s = 0; s < P.T; ++s) {
      const int t = P.T - 1 - s;
      clear();
      if (!top) {
        if (flags_above) wait_for(flags_above, s + 1);
        product(1, dp_above + (size_t)s * P.slot);
      }
      const Slopes slopes = node_slopes(gv, c_now, c_before);  // (off the chain)
      if (s > 0) {
        wait_for(flags_here, s);
        product(0, dp_here + (size_t)(s - 1) * P.slot);
      }
      float sum;
      if (!reduce(sum)) return abandon();
      const float other = __shfl_xor(sum, 1, 64);
      float next = s == 0 ? next0 : (seg == 0 ? sum : other), above = top ? top_v : (seg == 0 ? other : sum);
      if (P.clip > 0.0f) {
        next = clamp_error(next, P.clip);
        if (!top) above = clamp_error(above, P.clip);
      }
      float d[4];
      node_point(above + next, mask_v, slopes, ec, d);
      if (b < mb) {
        float* p = P.dp + (size_t)(l * (long long)P.T + s) * P.slot + dp_at;
        const float d0 = ok ? (seg ? d[2] : d[0]) : 0.0f, d1 = ok ? (seg ? d[3] : d[1]) : 0.0f;
        const unsigned long long v = (unsigned long long)__float_as_uint(d0) | (unsigned long long)__float_as_uint(d1) << 32;
        __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      zr_publish_barrier();
      if (tid == 0) __hip_atomic_store(flags_here + jt, s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (ok) {
        float* dg = P.dgates[l] + (size_t)t * 4 * n + (size_t)b * 4 * H + j;
        dg[(size_t)(2 * seg) * H] = seg ? d[2] : d[0];
        dg[(size_t)(2 * seg + 1) * H] = seg ? d[3] : d[1];
      }
      c_now = c_before;
      if (t > 0) fetch(t - 1);
    }
    // the error to the initial state
    clear();
    wait_for(flags_here, P.T);
    product(0, dp_here + (size_t)(P.T - 1) * P.slot);
    float sum;
    if (!reduce(sum)) return abandon();
    if (ok && seg == 0) {
      P.err_h0[l][ix] = P.clip > 0.0f ? clamp_error(sum, P.clip) : sum;
      P.err_c0[l][ix] = ec;
    }
  };
  work();

  // The last workgroup out returns the flags to zero for the next launch.
  zr_publish_barrier();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(P.departures, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == (int)gridDim.x - 1 ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;
  for (int i = tid; i < P.n_flags; i += 64 * kWaves) __hip_atomic_store(P.flags + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (tid == 0) __hip_atomic_store(P.departures, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The whole sweep of one column by one workgroup, where a launch above was abandoned.  The state between the steps lies in the launch's own
// hand-over memory, which nobody reads any more: per column [2][nl][H], the errors to h_{t-1} and to c_{t-1} (gate errors are in LDS).
__global__ void __launch_bounds__(512) lstm_backward_redo_kernel(BackResident P) {
  if (__hip_atomic_load(P.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != P.epoch) return;
  __shared__ float dg[4 * 512];
  const int b = blockIdx.x, tid = threadIdx.x, H = P.H;
  const size_t n = (size_t)H * P.mb, ix = (size_t)b * H + tid;
  const bool in = tid < H;  // (H <= 512)
  float* state = P.dp + (size_t)b * P.nl * 2 * H;
  float* err_h = state;                     // [nl][H] error to the step before
  float* ec = state + (size_t)P.nl * H;     // [nl][H]
  for (int l = 0; l < P.nl; ++l)
    if (in) {
      err_h[l * H + tid] = P.err_hT[l] ? P.err_hT[l][ix] : 0.0f;
      ec[l * H + tid] = P.err_cT[l] ? P.err_cT[l][ix] : 0.0f;
    }
  for (int t = P.T - 1; t >= 0; --t) {
    float above = in ? P.err_top[(size_t)t * n + ix] : 0.0f;
    const float m = (float)P.mask01[(size_t)t * P.mb + b];
    for (int l = P.nl - 1; l >= 0; --l) {
      if (in) {
        float next = err_h[l * H + tid], g[4], d[4], e = ec[l * H + tid];
        if (P.clip > 0.0f) {
          next = clamp_error(next, P.clip);
          if (l < P.nl - 1) above = clamp_error(above, P.clip);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) g[q] = P.gates[l][(size_t)(4 * t + q) * n + ix];
        node_point(above + next, m, node_slopes(g, P.c[l][(size_t)t * n + ix], t ? P.c[l][(size_t)(t - 1) * n + ix] : P.c0[l][ix]), e, d);
        ec[l * H + tid] = e;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          dg[q * H + tid] = d[q];
          P.dgates[l][(size_t)t * 4 * n + (size_t)b * 4 * H + q * H + tid] = d[q];
        }
      }
      __syncthreads();
      float to_h = 0.0f, to_below = 0.0f;
      if (in)
        for (int q0 = 0; q0 < 4 * H; q0 += 64) {  // (pieces: shorter chains of additions)
          float a = 0.0f, c = 0.0f;
          for (int q = q0; q < q0 + 64 && q < 4 * H; ++q) {
            a += P.stack[l][tid + (size_t)q * H] * dg[q];
            c += P.stack[l][tid + ((size_t)4 * H + q) * H] * dg[q];
          }
          to_h += a, to_below += c;
        }
      __syncthreads();
      if (in) err_h[l * H + tid] = to_h;
      above = to_below;
    }
    if (in && P.err_below0) P.err_below0[(size_t)t * n + ix] = above;
  }
  if (in)
    for (int l = 0; l < P.nl; ++l) {
      const float e = err_h[l * H + tid];
      P.err_h0[l][ix] = P.clip > 0.0f ? clamp_error(e, P.clip) : e;
      P.err_c0[l][ix] = ec[l * H + tid];
    }
}

typedef void (*Kernel)(BackResident);
constexpr int kClasses = ZR_BACK_CLASSES;
const Kernel kKernels[kClasses] = {lstm_backward_resident_kernel<4>, lstm_backward_resident_kernel<8>, lstm_backward_resident_kernel<10>,
                                   lstm_backward_resident_kernel<12>, lstm_backward_resident_kernel<16>};

int capacity(zr_ctx* ctx, int size_class) {
  int& cached = ctx->back_capacity[size_class];
  if (cached == 0) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kKernels[size_class], 64 * kWaves, 0) != hipSuccess) {
      (void)hipGetLastError();
      cached = -1;
    } else {
      cached = ctx->cu_count * per_cu > 0 ? ctx->cu_count * per_cu : -1;
    }
  }
  return cached > 0 ? cached : 0;
}

}  // namespace

ZrBackPlan zr_backward_resident_plan(zr_ctx* ctx, int nl, int H, int mb, int T, bool below) {
  ZrBackPlan plan = {};
  if (H < 8 || H > 512 || nl > kMaxLayers || T >= kGaveUp / 2) return plan;
  const int size_class = zr_back_size_class(H);
  if (64LL * ((H + 15) / 16) * ((mb + 7) / 8 * 8) * 4 >= 1LL << 32) return plan;
  return zr_back_plan(nl, H, mb, T, below, capacity(ctx, size_class), ZR_MAX_STEP_FLAGS - 32);
}

int zr_backward_resident_sweep(zr_ctx* ctx, const ZrBackPlan& plan, int nl, const float* const stacks[], int H, int T, int mb, const int* d_mask01,
                               const float* const d_c0[], const float* const d_c_all[], const float* const d_gates_all[], const float* d_err_top,
                               const float* const d_err_hT[], const float* const d_err_cT[], float* const d_dgates_all[], float* d_err_below0,
                               float* const d_err_h0[], float* const d_err_c0[], float err_clip) {
  BackResident P = {};
  P.j_tiles = (H + kRows - 1) / kRows;
  P.n_tiles = (mb + kCols - 1) / kCols;
  P.mbp = (mb + 7) / 8 * 8;
  P.slot = 64LL * P.j_tiles * P.mbp;
  void* p = nullptr;
  // (the redo kernel's state, 2 nl H floats a column, fits the slots of one step)
  const int rc = zr_ctx_scratch_if_room(ctx, 1, sizeof(float) * (size_t)((long long)nl * T * P.slot), &p);
  if (rc) return rc;
  for (int l = 0; l < nl; ++l) {
    P.stack[l] = stacks[l];
    P.gates[l] = d_gates_all[l];
    P.c[l] = d_c_all[l];
    P.c0[l] = d_c0[l];
    P.err_hT[l] = d_err_hT ? d_err_hT[l] : nullptr;
    P.err_cT[l] = d_err_cT ? d_err_cT[l] : nullptr;
    P.dgates[l] = d_dgates_all[l];
    P.err_h0[l] = d_err_h0[l];
    P.err_c0[l] = d_err_c0[l];
  }
  P.err_top = d_err_top;
  P.err_below0 = d_err_below0;
  P.mask01 = d_mask01;
  P.dp = (float*)p;
  P.flags = ctx->d_step_flags + 32;
  P.flag_stride = plan.flag_stride;
  P.departures = ctx->d_step_flags;
  P.failed = ctx->d_flags + 4;
  P.epoch = ctx->back_epoch = ctx->back_epoch % 0x7ffffff0 + 1;
  P.nl = nl;
  P.T = T;
  P.H = H;
  P.mb = mb;
  P.clip = err_clip;
  P.spin_limit = ctx->sweep_spin > 0 ? ctx->sweep_spin : (1 << 20);
  P.wait_extra = ctx->step_wait_extra;
  const int per = P.j_tiles * P.n_tiles;
  for (int left = nl; left > 0; left -= P.layers) {
    P.l_top = left - 1;
    P.layers = left < plan.at_once ? left : plan.at_once;
    P.below_parts = left == P.layers && plan.below && d_err_below0 ? 1 : 0;
    P.n_flags = P.layers * P.n_tiles * P.flag_stride;
    kKernels[plan.size_class]<<<(unsigned)((P.layers + P.below_parts) * per), 64 * kWaves, 0, ctx->stream>>>(P);
    ZR_LAUNCH_CHECK("lstm_backward_resident_kernel");
  }
  if (d_err_below0 && !plan.below) {  // in a launch of its own: its steps wait for nothing, so they are dealt out as well
    P.layers = P.n_flags = 0;
    P.below_parts = plan.capacity / per < T ? plan.capacity / per : T;
    kKernels[plan.size_class]<<<(unsigned)(P.below_parts * per), 64 * kWaves, 0, ctx->stream>>>(P);
    ZR_LAUNCH_CHECK("lstm_backward_resident_kernel");
  }
  lstm_backward_redo_kernel<<<mb, 512, 0, ctx->stream>>>(P);
  ZR_LAUNCH_CHECK("lstm_backward_redo_kernel");
  return ZR_OK;
}
