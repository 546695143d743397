// What zr_lstm.hip hands to the whole-sweep kernel (zr_lstm_sweep.hip).
#pragma once

#include "zr_internal.h"

constexpr int kMaxUnits = 8;           // layers of a sweep
constexpr int kSweepGaveUp = 1 << 28;  // bit set in every counter by a workgroup that stopped waiting
constexpr int kSweepCtrStride = 32;    // ints between counters: one 128-byte line each

struct LstmSweep {
  const float* W[kMaxUnits];     // per layer: [2][4] packed fp32 matrices
  const float* bias[kMaxUnits];  // per layer: [4][H]
  const float* h0[kMaxUnits];
  const float* c0[kMaxUnits];
  float* h_all[kMaxUnits];
  float* c_all[kMaxUnits];
  float* gates_all[kMaxUnits];   // null: gates not kept
  const float* embed;
  const int* ids;                // [T][mb], already non-negative
  const int* mask01;             // [T][mb]
  unsigned short* hp;            // [nl][T + 1] states of [3][H/8][columns][8]: h0 and every h as three bf16 terms
  unsigned short* xp;            // [T] states: the embedding columns the same way
  int* counters;                 // [nl][n_tiles] at kSweepCtrStride, zero at launch
  int* status;                   // set to 1 when a wait was abandoned
  int nl, T, V, H, mb, ldw, kp, j_tiles, n_tiles;
  float clip;
  int spin_limit;
  int columns;                   // mb rounded up to 8: no 128-byte line of the terms has two producers

  __device__ int clamp_id(int v) const { return v < 0 ? 0 : (v >= V ? V - 1 : v); }
};

// Resident workgroups of the kernel on tiles of 32 * tn columns that the device can hold at once (0: unknown / query failed).
int zr_sweep_capacity(zr_ctx* ctx, int tn);
// H a multiple of 8, T of at least 1; the counters are cleared, P.hp has its size, and the workgroups fit the device.
int zr_sweep_launch(zr_ctx* ctx, const LstmSweep& P, int tn);
