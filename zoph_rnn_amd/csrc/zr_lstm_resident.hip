// Whole stacked-LSTM sweep with the weights held in registers.
//
// lstm_sweep_kernel (zr_lstm.hip) streams every weight tile from the caches in every time step and gives a workgroup 32
// hidden rows: right when the batch is wide enough for the matrix cores to be the bound, but a small model or a narrow
// batch then runs on a handful of workgroups (H = 500, two layers: 32), each with a K loop far longer than the time
// step's arithmetic needs.  Here a workgroup owns 8 hidden rows of one layer -- 32 weight rows, its 8 rows of the four
// gates, the width of one matrix instruction -- for one column tile and all T steps, and its 8 waves keep their share of
// those 32 x 2H weights in vector registers: 2H x 32 floats over 512 threads is H/8 registers a thread, 128 at H = 1024.
// A time step then moves activations only.
//
// What bounds it: the chain of time steps -- h of (l, t-1) must be published by every row tile of the layer, seen by the
// others and multiplied before (l, t) can publish -- so everything that is not on that chain is kept off it:
//   * the product with the input from below (embedding columns, or h of (l-1, t), which is there a step early) runs
//     first, in the shadow of the hand-over of h of (l, t-1);
//   * a wave waits only for the producers of its own K slice: a row tile of 8 is one k-group, the flags of the 16
//     producers (at most) of a wave's groups lie side by side and one load by one wave looks at all of them;
//   * h travels in a k-interleaved copy [k/4][columns][4] whose pad rows are written as zeros (any H, no K tails) and
//     whose columns are padded to eight, so that every 128-byte line of it has one producer, with any number of column
//     tiles, and is read only after that producer's flag: no cache invalidation inside the launch (zr_resident_layout.h);
//   * h, c and the kept gate values are stored after the publish.
// Batches of up to 16 columns use the 16 x 16 x 4 instruction (NARROW), half the matrix time of a half-empty 32-column
// tile.  Progress, bounded waits and the abandon protocol are those of lstm_sweep_kernel; a workgroup that gives up marks
// its own flag, which makes everybody who depends on it give up in turn.  The last workgroup out clears the flags.
//
// Measured, whole sweep, against one launch per diagonal: 1 layer of H = 100, 8 columns, 20 steps 52 us (253); 2 of 500,
// 20 columns, 35 steps 169 us (1130); 4 of 1000, 50 steps, 16 columns 706 us (1575), 1 column 670 us (1520).
// Tried: finishing waves that publish on their own while the others run ahead into the next step (300 against 180 us at
// H = 500: the waves that are ahead poll, and their polls hold up the publishing stores); a first look at the flags of
// the layer below a step early (no change).
#include "zr_internal.h"
#include "zr_math.h"
#include "zr_mfma_core.h"
#include "zr_resident_layout.h"

namespace {

constexpr int kMaxLayers = 8;
constexpr int kWaves = 8;                 // waves per workgroup = K slices
constexpr int kRows = kResidentRows;
constexpr int kRedLd = 36;                // LDS row of 32 partial sums, padded: conflict-free for the cell's reads
constexpr int kResidentGaveUp = 1 << 28;  // flag value of a workgroup that stopped waiting

struct LstmResident {
  const float* W[kMaxLayers];     // per layer: [2][4] packed fp32 matrices
  const float* bias[kMaxLayers];  // per layer: [4][H]
  const float* h0[kMaxLayers];
  const float* c0[kMaxLayers];
  float* h_all[kMaxLayers];
  float* c_all[kMaxLayers];
  float* gates_all[kMaxLayers];   // null: gates not kept
  const float* embed;
  const int* ids;                 // [T][mb], already non-negative
  const int* mask01;              // [T][mb]
  float* hp;                      // [layers][T + 1] slots of k-interleaved h: slot 0 = initial state, slot t + 1 = h_t
  long long slot;                 // floats per slot (zr_resident_slot)
  int* flags;                     // [layers of this launch][n_tiles] at flag_stride, zero at launch: slots published
  int flag_stride, n_flags;
  int* departures;                // workgroups that have left the kernel (zero at launch)
  int* status;                    // set to 1 when a wait was abandoned
  int l_begin;                    // first layer of this launch (the layers below it are complete)
  int T, V, H, mb, mbp, ldw, kp, j_tiles, n_tiles;
  float clip;
  int spin_limit;
};

typedef zr_f32x4 zr_f32x4_u __attribute__((aligned(4)));  // 16-byte load from a 4-byte aligned address

// NG: k-groups per wave and segment (H <= 64 * NG, NARROW: 128 * NG).  TN: 32-column tiles per workgroup (NARROW: one
// 16-column tile).
template <int NG, int TN, bool NARROW>
__global__ void __launch_bounds__(64 * kWaves, NG * TN <= 4 ? 4 : 2) lstm_resident_kernel(LstmResident P) {
  static_assert(!NARROW || TN == 1, "a narrow tile is one tile of 16 columns");
  constexpr int KB = NARROW ? 4 : 2;             // k-blocks of 4 per k-group
  constexpr int NB = NARROW ? 2 : 1;             // 16-row halves of the 32 weight rows
  constexpr int COLS = NARROW ? 16 : 32 * TN;    // columns of the workgroup's tile
  constexpr int NPROD = NARROW ? 2 * NG : NG;    // producers of a wave's K slice
  constexpr int NOUT = (kRows * COLS + 511) / 512;  // (row, column) pairs a thread finishes
  // A long chain of fp32 additions rounds more than the schedule with one launch per diagonal, which divides K further.  So
  // the sums are taken in pieces: two accumulators, for even and odd k, in narrow tiles up to H = 256, whose registers
  // allow it; else the sums of CHAIN k-groups go to LDS and the accumulators start from zero again (wide tiles of H <= 256
  // have short chains as they are).  Error of h against 64 bits, one layer, 12 steps: H = 1024, 16 columns 3.9e-7 without, 2.2e-7
  // (2.4e-7 with one launch per diagonal), 512 3.0e-7, 2.3e-7 (2.4e-7), 1000 at 40 columns 3.9e-7, 2.7e-7 (3.0e-7).  Costs 0 to 2 %
  // of a sweep, 4 % at up to 4 columns of 256 < H <= 512.  (Two accumulators there: 12 %, for registers; the sums back from LDS
  // before the last group: 1.5 %.)
  constexpr int NACC = NARROW && NG <= 2 ? 2 : 1;
  constexpr bool PIECES = NG >= (NARROW ? 4 : 8);
  constexpr int CHAIN = NARROW ? 4 : 16;
  constexpr bool SUMS_AHEAD = !NARROW || NG > 4;  // the sums come back from LDS before the last group
  __shared__ float red[kWaves * COLS * kRedLd + kRows];  // (the last rows: read, not used, by threads that publish zeros)
  __shared__ float s_bias[4][kRows];  // (registers are short)
  __shared__ int s_abort, s_last;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int kslice = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = P.H, mb = P.mb;
  const int nt = (int)blockIdx.x % P.n_tiles;
  const int jt = ((int)blockIdx.x / P.n_tiles) % P.j_tiles;
  const int l = P.l_begin + (int)blockIdx.x / (P.n_tiles * P.j_tiles);
  const int j0 = jt * kRows;
  const int n0 = nt * COLS;
  const int cl = NARROW ? (lane & 15) : (lane & 31);  // this lane's column of the activations, row of the weights
  const int kq = NARROW ? (lane >> 4) : (lane >> 5);  // its k-block inside a group
  const bool from_embed = l == 0;
  if (tid == 0) s_abort = 0;

  auto work = [&]() {
    // ---- weights into registers: w[segment][group][half][k]
    float w[2][NG][NB][4];
    const long long HH = (long long)P.kp * P.ldw;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NG; ++i)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int c = cl + 16 * b;
          const float* m = P.W[l] + (s * 4 + (c >> 3)) * HH + 4 * (j0 + (c & 7));
          const int k0 = 4 * (KB * (kslice + kWaves * i) + kq);
          if (s == 0 && from_embed && 4 * KB * (kslice + kWaves * i + 1) > H - 4) {  // uniform
            // Embedding columns are read as they lie, so a lane's four k must stay inside the column: k-blocks that reach
            // past its end, or lie behind it, are moved down to end at H - 1.  Every place that reads the same k keeps a part
            // of its weight: not zero in all but one, for zero times an infinite activation is not zero.
            const int ks = k0 < H - 4 ? k0 : H - 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int k = ks + e;
              w[s][i][b][e] = ldexpf(m[(long long)(k >> 2) * (4 * P.ldw) + (k & 3)],
                                     -zr_resident_embed_halvings(H, NG * kWaves * KB, k0 >> 2, k));
            }
          } else {
            zr_f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (k0 < P.kp) v = *(const zr_f32x4*)(m + (long long)(k0 >> 2) * (4 * P.ldw));
#pragma unroll
            for (int e = 0; e < 4; ++e) w[s][i][b][e] = v[e];
          }
        }

    // ---- the outputs this thread finishes: (row, column) pairs, rows of four fastest (the order h travels in).  A narrow
    // k-group is two row tiles: behind an odd number of them the last one's workgroup also publishes a tile of zeros.
    const int publishes = (NARROW && (P.j_tiles & 1) && jt == P.j_tiles - 1 ? 2 : 1) * kRows * COLS;
    int oj[NOUT], on[NOUT];
    bool ok[NOUT], tile_ok[NOUT];
    float c_state[NOUT];
    if (tid < 4 * kRows)  // (shifts and masks: a remainder of a signed index costs two registers, and those a tenth of a step)
      (&s_bias[0][0])[tid] = P.bias[l][(tid >> 3) * H + (j0 + (tid & 7) < H ? j0 + (tid & 7) : H - 1)];
    unsigned hp_off[NOUT];  // element inside a slot
#pragma unroll
    for (int u = 0; u < NOUT; ++u) {
      const int o = tid + 512 * u;
      oj[u] = ((o >> 2) / COLS) * 4 + (o & 3);
      on[u] = (o >> 2) % COLS;
      const int j = j0 + oj[u], n = n0 + on[u];
      tile_ok[u] = o < publishes && n < mb;
      ok[u] = tile_ok[u] && j < H;
      const int jc = j < H ? j : H - 1, nc = n < mb ? n : mb - 1;
      c_state[u] = P.c0[l][(long long)nc * H + jc];
      hp_off[u] = zr_resident_at(j, n, P.mbp);
    }
    int* flags_here = P.flags + ((l - P.l_begin) * P.n_tiles + nt) * P.flag_stride;
    const int* flags_below = flags_here - P.n_tiles * P.flag_stride;
    // Flags of a (layer, column tile): [K slice][producer of the slice].
    int pslice, pindex;  // where this workgroup stands as a producer
    if constexpr (NARROW)
      pslice = (jt >> 1) & 7, pindex = (jt >> 4) * 2 + (jt & 1);
    else
      pslice = jt & 7, pindex = jt >> 3;
    int* my_flag = flags_here + pslice * NPROD + pindex;
    // the producer this lane looks at, for the lanes below NPROD
    const int pj = NARROW ? 2 * (kslice + kWaves * (lane >> 1)) + (lane & 1) : kslice + kWaves * lane;
    const bool looks = lane < NPROD && pj < P.j_tiles;
    const int look = kslice * NPROD + (lane < NPROD ? lane : 0);
    bool dead = false;  // this wave has given up a wait: it goes on without waiting to the next barrier
    auto wait_for = [&](const int* flags, int target) {
      if (dead) return;
      int spins = 0;
      bool gave_up = false;
      for (;;) {
        const int v =
            looks ? __hip_atomic_load(flags + look, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : kResidentGaveUp - 1;
        if (__all(v >= target)) {
          gave_up = __any(v >= kResidentGaveUp);
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

    // ---- the initial state goes out as slot 0
    float* hp_mine = P.hp + (long long)l * (P.T + 1) * P.slot;
    const float* hp_below = hp_mine - (long long)(P.T + 1) * P.slot;
#pragma unroll
    for (int u = 0; u < NOUT; ++u)
      if (tile_ok[u])
        __hip_atomic_store(hp_mine + hp_off[u], ok[u] ? P.h0[l][(long long)(n0 + on[u]) * H + j0 + oj[u]] : 0.0f,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    zr_publish_barrier();
    if (tid == 0) __hip_atomic_store(my_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // ---- this lane's activation columns
    int cols[TN], idv[TN];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int c = n0 + tn * 32 + cl;
      cols[tn] = c < mb ? c : mb - 1;
    }
    auto clamp_id = [&](int v) { return v < 0 ? 0 : (v >= P.V ? P.V - 1 : v); };
    // The embedding columns of a step's words, read as they lie.  AHEAD: a step ahead (H = 1000, 16 columns: 6.8 us a step
    // against 7.5; no gain at smaller sizes, whose shorter segments leave nothing to hide the earlier loads behind).
    constexpr bool AHEAD = NARROW && NG == 8;
    zr_f32x4 x_ahead[AHEAD ? NG : 1][TN];
    const float* col[TN];
    auto next_words = [&](int t) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        col[tn] = P.embed + (long long)idv[tn] * H;
        idv[tn] = clamp_id(P.ids[(long long)(t + 1 < P.T ? t + 1 : t) * mb + cols[tn]]);
      }
    };
    auto load_embed = [&](zr_f32x4 (&x)[TN], int i) {
      const int k0 = 4 * (KB * (kslice + kWaves * i) + kq);
      const int ks = k0 < H - 4 ? k0 : H - 4;
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) x[tn] = *(const zr_f32x4_u*)(col[tn] + ks);
    };
    if (from_embed) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) idv[tn] = clamp_id(P.ids[cols[tn]]);
      next_words(0);
      if constexpr (AHEAD) {
#pragma unroll
        for (int i = 0; i < NG; ++i) load_embed(x_ahead[i], i);
      }
    }
    const unsigned kb_step = (unsigned)(kWaves * KB * P.mbp * 4);  // elements from a wave's group to its next
    const unsigned kb_first = (unsigned)((KB * kslice + kq) * P.mbp * 4);
    // Groups past the end are not read at all: a line read before its producer's flag would go stale.
    const int n_groups = (2 * P.j_tiles + KB - 1) / KB;

    typedef float acc16 __attribute__((ext_vector_type(16)));
    for (int t = 0; t < P.T; ++t) {
      acc16 acc[TN];
      zr_f32x4 acc4[NACC][NB];
      auto clear = [&]() {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[tn][r] = 0.0f;
#pragma unroll
        for (int q = 0; q < NACC; ++q)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc4[q][b] = {0.0f, 0.0f, 0.0f, 0.0f};
      };
      clear();
      // Partial sum u of this lane, and its place in LDS (the wave's own; free since the barrier behind the last cell).
      constexpr int NE = NARROW ? 4 * NB : 16 * TN;
      auto element = [&](int u) -> float {
        if constexpr (!NARROW)
          return acc[u >> 4][u & 15];
        else if constexpr (NACC == 2)
          return acc4[0][u >> 2][u & 3] + acc4[1][u >> 2][u & 3];
        else
          return acc4[0][u >> 2][u & 3];
      };
      float* mine = red + kslice * (COLS * kRedLd) + 4 * kq * kRedLd + cl;
      auto place = [&](int u) -> float& {
        return NARROW ? mine[(u & 3) * kRedLd + 16 * (u >> 2)] : mine[((u >> 4) * 32 + 8 * ((u >> 2) & 3) + (u & 3)) * kRedLd];
      };
      float before[PIECES ? NE : 1];  // the sums of all but the last chain
      auto mma = [&](int seg, int i, const zr_f32x4 (&x)[TN], const float (&wg)[NB][4]) {
        if (PIECES && SUMS_AHEAD && seg == 1 && i == NG - 1) {  // on their way while the last group is multiplied
#pragma unroll
          for (int u = 0; u < NE; ++u) before[PIECES ? u : 0] = place(u);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (NARROW) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              zr_f32x4& a = acc4[e & (NACC - 1)][b];
              a = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0][e], wg[b][e], a, 0, 0, 0);
            }
          } else {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
              acc[tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[tn][e], wg[0][e], acc[tn], 0, 0, 0);
          }
        }
        if (PIECES && ((i + 1) % CHAIN == 0 || i == NG - 1) && !(seg == 1 && i == NG - 1)) {
#pragma unroll
          for (int u = 0; u < NE; ++u) place(u) = seg == 0 && i < CHAIN ? element(u) : place(u) + element(u);
          clear();
        }
      };
      // One segment.  All of a wave's activations are in flight at once where the registers allow it, else a few groups
      // ahead of the ones being multiplied.
      auto segment = [&](int seg, auto load) {
        constexpr int CH = NG <= 8 ? NG : (TN == 1 ? 4 : 2);
        constexpr int NC = NG / CH;
        zr_f32x4 x[NC > 1 ? 2 : 1][CH][TN];
#pragma unroll
        for (int i = 0; i < CH; ++i) load(x[0][i], i);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (c + 1 < NC) {
#pragma unroll
            for (int i = 0; i < CH; ++i) load(x[(c + 1) & (NC > 1 ? 1 : 0)][i], (c + 1) * CH + i);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < CH; ++i) mma(seg, c * CH + i, x[c & (NC > 1 ? 1 : 0)][i], w[seg][c * CH + i]);
        }
      };
      auto load_packed = [&](const float* base) {
        return [=, &cols](zr_f32x4 (&x)[TN], int i) {
          if (kslice + kWaves * i < n_groups) {
            const unsigned kb = kb_first + (unsigned)i * kb_step;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) x[tn] = *(const zr_f32x4*)(base + (kb + 4u * (unsigned)cols[tn]));
          } else {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) x[tn] = zr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
        };
      };

      // the input from below
      if (from_embed) {
        if constexpr (AHEAD) {
#pragma unroll
          for (int i = 0; i < NG; ++i) mma(0, i, x_ahead[i], w[0][i]);
        } else {
          segment(0, load_embed);
        }
      } else {
        if (l > P.l_begin) wait_for(flags_below, t + 2);
        segment(0, load_packed(hp_below + (long long)(t + 1) * P.slot));
      }
      float mask_v[NOUT];
#pragma unroll
      for (int u = 0; u < NOUT; ++u) mask_v[u] = tile_ok[u] ? (float)P.mask01[(long long)t * mb + n0 + on[u]] : 0.0f;
      // the layer's own previous step
      wait_for(flags_here, t + 1);
      segment(1, load_packed(hp_mine + (long long)t * P.slot));

      // what the next step reads from below: asked for now, in flight while this step is finished
      if (t + 1 < P.T) {
        if (from_embed) {
          next_words(t + 1);
          if constexpr (AHEAD) {
#pragma unroll
            for (int i = 0; i < NG; ++i) load_embed(x_ahead[i], i);
          }
        }
      }

      // partial sums of the 8 K slices through LDS, then the cell
#pragma unroll
      for (int u = 0; u < NE; ++u) place(u) = !PIECES ? element(u) : (SUMS_AHEAD ? before[PIECES ? u : 0] : place(u)) + element(u);
      __syncthreads();
      if (s_abort) {  // every wave of the workgroup sees the same value: waits come before this barrier
        if (tid == 0) __hip_atomic_store(my_flag, kResidentGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tid == 0) __hip_atomic_store(P.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
      float h_v[NOUT], g_v[NOUT][4];
      float* hp_out = hp_mine + (long long)(t + 1) * P.slot;
#pragma unroll
      for (int u = 0; u < NOUT; ++u) {
        if (!tile_ok[u]) continue;
        float z[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float* p = red + on[u] * kRedLd + g * 8 + oj[u];
          float part[kWaves];
#pragma unroll
          for (int q = 0; q < kWaves; ++q) part[q] = p[q * (COLS * kRedLd)];
          z[g] = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        }
        float c;
        const int row = oj[u] & (kRows - 1);  // (a tile of zeros has rows past the tile)
        zr_lstm_cell(z[0] + s_bias[0][row], z[1] + s_bias[1][row], z[2] + s_bias[2][row], z[3] + s_bias[3][row], c_state[u], mask_v[u], P.clip, g_v[u][0],
                     g_v[u][1], g_v[u][2], g_v[u][3], c, h_v[u]);
        c_state[u] = c;
        __hip_atomic_store(hp_out + hp_off[u], ok[u] ? h_v[u] : 0.0f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      zr_publish_barrier();
      if (tid == 0) __hip_atomic_store(my_flag, t + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < NOUT; ++u) {
        if (!ok[u]) continue;
        const long long n_el = (long long)H * mb;
        const long long ix = (long long)(n0 + on[u]) * H + j0 + oj[u];
        P.h_all[l][(long long)t * n_el + ix] = h_v[u];
        P.c_all[l][(long long)t * n_el + ix] = c_state[u];
        if (P.gates_all[l]) {
          float* gt = P.gates_all[l] + (long long)t * 4 * n_el + ix;
#pragma unroll
          for (int g = 0; g < 4; ++g) gt[g * n_el] = g_v[u][g];
        }
      }
    }
  };
  __syncthreads();  // s_abort
  work();

  // Departure: the last workgroup out returns the flags to zero for the next launch (this one's own last flag has
  // landed by then).
  zr_publish_barrier();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(P.departures, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == (int)gridDim.x - 1 ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;
  for (int i = tid; i < P.n_flags; i += 512) __hip_atomic_store(P.flags + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (tid == 0) __hip_atomic_store(P.departures, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

typedef void (*ResidentKernel)(LstmResident);
// [size class][column class]: H <= 128, 256, 512, 1024; 16, 32, 64 columns a workgroup (64 columns of H > 512: the
// registers hold 128 weights a thread and not the 32 accumulators on top)
const ResidentKernel kKernels[4][3] = {
    {lstm_resident_kernel<1, 1, true>, lstm_resident_kernel<2, 1, false>, lstm_resident_kernel<2, 2, false>},
    {lstm_resident_kernel<2, 1, true>, lstm_resident_kernel<4, 1, false>, lstm_resident_kernel<4, 2, false>},
    {lstm_resident_kernel<4, 1, true>, lstm_resident_kernel<8, 1, false>, lstm_resident_kernel<8, 2, false>},
    {lstm_resident_kernel<8, 1, true>, lstm_resident_kernel<16, 1, false>, nullptr}};

int resident_capacity(zr_ctx* ctx, int size_class, int col_class) {
  int& cached = ctx->resident_capacity[size_class][col_class];
  if (!kKernels[size_class][col_class]) return 0;
  if (cached == 0) {
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kKernels[size_class][col_class], 64 * kWaves, 0) != hipSuccess) {
      (void)hipGetLastError();
      cached = -1;
    } else {
      ctx->cu_count = cus;
      cached = cus * per_cu > 0 ? cus * per_cu : -1;
    }
  }
  return cached > 0 ? cached : 0;
}

}  // namespace

ZrResidentPlan zr_lstm_resident_plan(zr_ctx* ctx, int nl, int H, int mb, int T) {
  ZrResidentPlan plan = {};
  plan.us = -1.0;
  if (H < 8 || H > 1024 || nl > kMaxLayers || T >= kResidentGaveUp / 2) return plan;
  if (zr_resident_slot(H, mb) * 4 >= (1LL << 32)) return plan;
  const int size_class = H <= 128 ? 0 : (H <= 256 ? 1 : (H <= 512 ? 2 : 3));
  int capacity[3];
  for (int c = 0; c < 3; ++c) capacity[c] = resident_capacity(ctx, size_class, c);
  return zr_sweep_resident_plan(nl, H, mb, T, capacity, ZR_MAX_STEP_FLAGS - 32, ctx->cu_count);
}

int zr_lstm_resident_sweep(zr_ctx* ctx, const ZrResidentPlan& plan, int nl, const zr_lstm_weights* const layers[],
                           const float* d_embed, int V, const int* d_ids_nonneg, const int* d_mask01, int T, int mb,
                           const float* const d_h0[], const float* const d_c0[], float clip_threshold,
                           float* const d_h_all[], float* const d_c_all[], float* const d_gates_all[]) {
  const int H = layers[0]->H;
  const int j_tiles = (H + kRows - 1) / kRows;
  const int per_layer = j_tiles * plan.n_tiles;
  const long long slot = zr_resident_slot(H, mb);
  void* p = nullptr;
  int rc = zr_ctx_scratch_if_room(ctx, 1, sizeof(float) * (size_t)(nl * (long long)(T + 1) * slot), &p);
  if (rc) return rc;
  LstmResident P = {};
  for (int l = 0; l < nl; ++l) {
    P.W[l] = (const float*)layers[l]->d_W;
    P.bias[l] = layers[l]->d_bias;
    P.h0[l] = d_h0[l];
    P.c0[l] = d_c0[l];
    P.h_all[l] = d_h_all[l];
    P.c_all[l] = d_c_all[l];
    P.gates_all[l] = d_gates_all ? d_gates_all[l] : nullptr;
  }
  P.embed = d_embed;
  P.ids = d_ids_nonneg;
  P.mask01 = d_mask01;
  P.hp = (float*)p;
  P.slot = slot;
  P.flags = ctx->d_step_flags + 32;
  P.flag_stride = plan.flag_stride;
  P.departures = ctx->d_step_flags;
  P.status = ctx->d_flags + 2;
  P.T = T;
  P.V = V;
  P.H = H;
  P.mb = mb;
  P.mbp = zr_resident_columns(mb);
  P.ldw = layers[0]->ldw;
  P.kp = layers[0]->kp;
  P.j_tiles = j_tiles;
  P.n_tiles = plan.n_tiles;
  P.clip = clip_threshold;
  P.spin_limit = ctx->sweep_spin > 0 ? ctx->sweep_spin : (1 << 20);
  for (int l = 0; l < nl; l += plan.at_once) {
    const int now = nl - l < plan.at_once ? nl - l : plan.at_once;
    P.l_begin = l;
    P.n_flags = now * plan.n_tiles * plan.flag_stride;
    kKernels[plan.size_class][plan.col_class]<<<now * per_layer, 64 * kWaves, 0, ctx->stream>>>(P);
    ZR_LAUNCH_CHECK("lstm_resident_kernel");
  }
  return ZR_OK;
}
