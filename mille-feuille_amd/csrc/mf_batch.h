// mf_batch.h -- work items and arguments of the batched CG kernels.
#pragma once

#include "mf_strips.h"

namespace mf {

// Waves per (system, right-hand side) item: 4, 8 or 16, picked by
// opts->batch_waves or by mf_tune_batch.
struct BatchSys {
  TileView A;
  StripView S;         // strip kernel
  const int *wave_tr;  // tile kernel: waves per item + 1 tile-row bounds
  const double *b;     // npad * nrhs, right-hand side j at j * npad
  double *x;           // npad * nrhs
  int npad;
  int mixed;           // 1: per-tile levels (A.prec), 0: every tile FP64
};

struct BatchArgs {
  const BatchSys *sys;
  const int2 *items;  // (system, right-hand side), queue by queue
  const int *qoff;    // kQueues + 1: items of queue q at [qoff[q], qoff[q+1])
  int nitems;
  int *head;          // kQueues work-queue heads
  double *work;       // per block: r, p, q (npad_max doubles each), p32
  long long stride;   // doubles per block
  int npad_max;       // longest vector of the batch
  int *iters;
  double *relres;
  unsigned long long *tstamp;  // per item: start, end
  double tol2;
  int maxiter;
  double ratio2;
  int max_refresh;
  int refresh_every;
};

constexpr int kQueues = 8;  // one per XCD

__device__ __forceinline__ unsigned long long realtime() { return __builtin_amdgcn_s_memrealtime(); }

// Next item of the block's queue q, -1 when every queue is empty: an empty
// queue passes to the next one, and after all kQueues the block ends (every
// head only grows).  One thread.
__device__ __forceinline__ int next_item(const BatchArgs &a, int &q, int &tried) {
  while (tried < kQueues) {
    const int k = atomicAdd(&a.head[q], 1);
    if (a.qoff[q] + k < a.qoff[q + 1]) return a.qoff[q] + k;
    q = (q + 1) % kQueues;
    ++tried;
  }
  return -1;
}

// Strip kernel for `waves` waves per item.
const void *batch_strip_kernel(int waves, bool mixed);

}  // namespace mf
