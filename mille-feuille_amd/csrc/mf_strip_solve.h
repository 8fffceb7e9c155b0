// mf_strip_solve.h -- arguments of the strip solvers and their host entry.
#pragma once

#include "mf_strips.h"

namespace mf {

enum StatSlot {
  kStIters = 0,
  kStRefresh,
  kStFallback,
  kStRecursive,
  kStTrue,
  kStBB,
  kStStatus,
  kStCount = 16
};

constexpr int kBlock = 1024;  // 16 waves, one block per CU
constexpr int kWavesPerBlock = kBlock / 64;
// Strips per wave whose vectors a strip solver holds in registers.
constexpr int kMaxWaveStrips = 8;

struct StripSolveArgs {
  StripView S;
  TileView A;                // tile levels (learned policy, histogram)
  const double *b;
  double *x;
  double *r, *p;             // vectors in memory, FP64 (r: BiCGSTAB's s) ...
  float *r32, *p32;          // ... and FP32 (mixed)
  const int *wave_piece;     // per wave, bounds of its pieces in piece_order
  const int *piece_order;
  unsigned long long *pmail; // two tagged words per piece
  double *partials;
  unsigned long long *mbox;
  GridSync *gs;
  double *stats;
  unsigned long long *hist;
  double tol2, ratio2;
  int maxiter, fixed_iters, check_interval, max_refresh, refresh_every;
  const MlpDevice *mlp;      // learned policy, else null
  const uint16_t *feat16;
  float *seg2;
  uint8_t *prec_rw;
  int nseg;
};

// Kernel of the strip CG or BiCGSTAB for `strips` strips per wave (1 ..
// kMaxWaveStrips).
const void *strip_solve_kernel(int strips, bool bicg, bool mixed);

}  // namespace mf
