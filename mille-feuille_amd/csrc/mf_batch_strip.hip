// mf_batch_strip.hip -- batched CG over row strips: one block solves one
// (system, right-hand side) item, with textbook CG (as k_batch_cg), queues,
// refreshes and fallback of mf_batch.hip.
//
// A system of at most NW * KB strips (a wave holds KB strips' rows) keeps its
// vectors on chip for the whole solve: the search direction p in LDS, where
// the product gathers it, q = A p in LDS, r and x in registers; only the
// matrix is read per iteration, through the XCD's L2, which the blocks that
// solve the system's other right-hand sides share.  KB is 8 for FP64 vectors
// and 16 for FP32 ones: 16 waves hold 8,192 or 16,384 rows in 128 KB of LDS.
// Larger systems keep the vectors in the block's workspace in memory.
//
// Mixed items multiply the FP32 payload with FP32 r, p and q (x, scalars and
// residual recomputations FP64); a stagnating one goes on in FP64, from its
// x, with the vectors in memory.
//
// Measured on MI355X, 48 kNN systems of 1,000 to 16,000 rows x 8 right-hand
// sides: error bound 12.0 ms (k_batch_cg 54), FP64 18.9 ms; the largest system
// sets the time, 39.6 us an iteration on its CU (155 before), 69 with the
// vectors in memory (FP64).  What is left is the matrix: 16 strips a wave, two
// trips through the L2 each.
#include <cmath>
#include <type_traits>

#include "mf_batch.h"

namespace mf {

namespace {

// Strip k of wave w: the waves take strips in turns of alternating order, so
// that in sorted layouts (longest rows first in every window) none gets the
// long ones each time.
template <int NW>
__device__ __forceinline__ int wave_strip(int w, int k) {
  return NW * k + (k & 1 ? NW - 1 - w : w);
}

// A x over the block: pieces of long rows first (sums to part), then
// f(strip, row, sum, own entry of x) for every strip lane with a row.  The
// caller's vectors are complete on entry; a block barrier follows before the
// next product.
template <int NW, class X, class F>
__device__ __forceinline__ void block_product(const StripView &S, int w, int lane, const X &x, bool v32, double *part,
                                              F f) {
  if (S.npieces > 0) {
    for (int q = w; q < S.npieces; q += NW) {
      const double v = piece_sum(S, q, lane, x, v32);
      if (lane == 0) part[q] = v;
    }
    __syncthreads();
  }
  int n = (S.nstrips + NW - 1) / NW;
  if (n > 0 && wave_strip<NW>(w, n - 1) >= S.nstrips) --n;
  strips_run<false>(S, lane, x, v32, n, [&](int k) { return wave_strip<NW>(w, k); },
             [&](int s, const StripDesc &d, int row, bool lng, double acc, double own) {
               if ((d.flags & kStripLong) && lng) {
                 const LongRow lr = S.lrow[S.lane_long[64 * s + lane]];
                 for (int j = 0; j < lr.n; ++j) acc += part[lr.first + j];
               }
               if (row >= 0) f(s, row, acc, own);
             });
}

struct ItemState {
  double bb = 0.0, stop2 = 0.0, rr = 0.0, rr_ref = 0.0;
  int it = 0, it_ref = 0, refresh = 0;
};

enum ItemEnd { kItemDone, kItemNeeds64 };

// What to do with a recomputed residual tr (rr_new: the recursive one).
enum AfterRefresh { kGoOn, kStop, kFallBack, kRestart };
template <bool MIXED>
__device__ __forceinline__ AfterRefresh after_refresh(const BatchArgs &a, ItemState &st, double tr, double rr_new) {
  ++st.refresh;
  st.it_ref = st.it;
  if (tr <= st.stop2) {
    st.rr = tr;
    return kStop;
  }
  if (MIXED && (tr > 0.25 * st.rr_ref || st.refresh > a.max_refresh)) return kFallBack;
  st.rr_ref = tr;
  return tr > 4.0 * rr_new ? kRestart : kGoOn;
}

// CG with the vectors on chip.  lp: p by row; lq: A times the vector, by strip
// lane.  Each round is one product: of x for a residual, or of p.  Returns
// with x in memory.
template <int NW, int KB, typename VT>
__device__ __forceinline__ ItemEnd item_on_chip(const BatchArgs &a, const StripView &S, const double *b, double *gx,
                                                VT *lp, VT *lq, double *part, double *lds, ItemState &st) {
  constexpr bool MIXED = std::is_same<VT, float>::value;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows of the wave's strips (0xffff: none), two to a register
  uint32_t rows[KB / 2];
  VT r[KB];
  double x[KB];
  // (both hidden from the optimizer, which would otherwise keep every strip's
  // addresses in registers for the whole solve)
  auto row_of = [&](int k) {
    uint32_t v = rows[k / 2];
    asm("" : "+v"(v));
    v = k & 1 ? v >> 16 : v & 0xffffu;
    return v == 0xffffu ? -1 : (int)v;
  };
  auto slot = [&](int k) {
    int l = lane;
    asm("" : "+v"(l));
    return 64 * wave_strip<NW>(w, k) + l;
  };
#pragma unroll
  for (int k = 0; k < KB; ++k) {
    const int s = wave_strip<NW>(w, k);
    bool lng;
    const int i = s < S.nstrips ? strip_row(S, s, lane, lng) : -1;
    rows[k / 2] = (k & 1 ? rows[k / 2] : 0u) | (uint32_t)(i & 0xffff) << (16 * (k & 1));
    x[k] = i >= 0 ? gx[i] : 0.0;
    r[k] = VT(0);
  }
  double alpha = 0.0, beta = 0.0, rr = 0.0, rr_new = 0.0;
  bool res = true, init = true, stop = false;
  for (;;) {
    double pq0 = 0.0;
    if (res)
      block_product<NW>(S, w, lane, MemVec<double>{gx}, false, part,
                        [&](int s, int i, double v, double) { lq[64 * s + lane] = (VT)(b[i] - v); });
    else
      block_product<NW>(S, w, lane, LdsVec<VT>{lp}, MIXED, part, [&](int s, int, double v, double own) {
        lq[64 * s + lane] = (VT)v;
        pq0 += own * v;
      });
    bool restart = false;
    if (res) {
      double s2 = 0.0;
#pragma unroll
      for (int k = 0; k < KB; ++k)
        if (row_of(k) >= 0) {
          r[k] = lq[slot(k)];
          s2 += (double)r[k] * (double)r[k];
        }
      const double tr = block_sum(s2, lds);
      res = false;
      if (init) {
        init = false;
        rr = st.rr = st.rr_ref = tr;
        if (tr <= st.stop2) return kItemDone;
        restart = true;
      } else {
        const AfterRefresh go = after_refresh<MIXED>(a, st, tr, rr_new);
        if (go == kStop) return kItemDone;
        if (go == kFallBack && st.it < a.maxiter) return kItemNeeds64;
        if (go == kRestart) {
          restart = true;
          ++st.refresh;
        }
        beta = tr / rr;
        st.rr = rr = tr;
        if (st.it >= a.maxiter) return kItemDone;
      }
    } else {
      const double pq = block_sum(pq0, lds);
      stop = !(pq != 0.0) || !isfinite(pq) || (MIXED && !(pq > 0.0));
      if (!stop) {
        alpha = rr / pq;
        double rn = 0.0;
#pragma unroll
        for (int k = 0; k < KB; ++k)
          if (const int i = row_of(k); i >= 0) {
            x[k] += alpha * (double)lp[i];
            r[k] = (VT)((double)r[k] - alpha * (double)lq[slot(k)]);
            rn += (double)r[k] * (double)r[k];
          }
        rr_new = block_sum(rn, lds);
        res = rr_new <= st.stop2 ||
              (MIXED && (rr_new <= a.ratio2 * st.rr_ref || st.it - st.it_ref >= a.refresh_every));
      }
      if (stop || res || st.it >= a.maxiter) {
        // x to memory, for the residual or as the result
#pragma unroll
        for (int k = 0; k < KB; ++k)
          if (const int i = row_of(k); i >= 0) gx[i] = x[k];
        __syncthreads();
        if (stop) return MIXED ? kItemNeeds64 : kItemDone;
        if (res) continue;
      }
      beta = rr_new / rr;
      st.rr = rr = rr_new;
      if (st.it >= a.maxiter) return kItemDone;
    }
    // p = r + beta p (restart: p = r)
#pragma unroll
    for (int k = 0; k < KB; ++k)
      if (const int i = row_of(k); i >= 0) {
        const double po = restart ? 0.0 : (double)lp[i];
        lp[i] = (VT)((double)r[k] + beta * po);
      }
    __syncthreads();
    ++st.it;
  }
}

// CG with the vectors r, p, q in the block's workspace.
template <int NW, typename VT>
__device__ __forceinline__ ItemEnd item_in_memory(const BatchArgs &a, const StripView &S, const double *b, double *x,
                                                  double *work, int npad, double *part, double *lds, ItemState &st) {
  constexpr bool MIXED = std::is_same<VT, float>::value;
  constexpr int BLOCK = 64 * NW;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  VT *r = (VT *)work, *p = (VT *)(work + npad), *q = (VT *)(work + 2 * (size_t)npad);
  // gathered entries past the rows
  for (int i = S.nrows + threadIdx.x; i < npad; i += BLOCK) p[i] = VT(0);
  double beta = 0.0, rr = 0.0, rr_new = 0.0;
  bool res = true, init = true;
  for (;;) {
    double sum0 = 0.0;
    if (res)
      block_product<NW>(S, w, lane, MemVec<double>{x}, false, part, [&](int, int i, double v, double) {
        const VT rv = (VT)(b[i] - v);
        r[i] = rv;
        sum0 += (double)rv * (double)rv;
      });
    else
      block_product<NW>(S, w, lane, MemVec<VT>{p}, MIXED, part, [&](int, int i, double v, double own) {
        q[i] = (VT)v;
        sum0 += own * v;
      });
    const double sum = block_sum(sum0, lds);
    bool restart = false;
    if (res) {
      res = false;
      if (init) {
        init = false;
        rr = st.rr = st.rr_ref = sum;
        if (sum <= st.stop2) return kItemDone;
        restart = true;
      } else {
        const AfterRefresh go = after_refresh<MIXED>(a, st, sum, rr_new);
        if (go == kStop) return kItemDone;
        if (go == kFallBack && st.it < a.maxiter) return kItemNeeds64;
        if (go == kRestart) {
          restart = true;
          ++st.refresh;
        }
        beta = sum / rr;
        st.rr = rr = sum;
        if (st.it >= a.maxiter) return kItemDone;
      }
    } else {
      if (!(sum != 0.0) || !isfinite(sum) || (MIXED && !(sum > 0.0))) return MIXED ? kItemNeeds64 : kItemDone;
      const double alpha = rr / sum;
      double rn = 0.0;
      for (int i = threadIdx.x; i < S.nrows; i += BLOCK) {
        x[i] += alpha * (double)p[i];
        const VT rv = (VT)((double)r[i] - alpha * (double)q[i]);
        r[i] = rv;
        rn += (double)rv * (double)rv;
      }
      rr_new = block_sum(rn, lds);
      res = rr_new <= st.stop2 ||
            (MIXED && (rr_new <= a.ratio2 * st.rr_ref || st.it - st.it_ref >= a.refresh_every));
      if (res) continue;  // (the sum's barriers completed x)
      beta = rr_new / rr;
      st.rr = rr = rr_new;
      if (st.it >= a.maxiter) return kItemDone;
    }
    for (int i = threadIdx.x; i < S.nrows; i += BLOCK)
      p[i] = restart ? r[i] : (VT)((double)r[i] + beta * (double)p[i]);
    __syncthreads();
    ++st.it;
  }
}

}  // namespace

template <int NW, bool MIXED>
__global__ __launch_bounds__(64 * NW, 4) void k_batch_strip(BatchArgs a) {
  using VT = typename std::conditional<MIXED, float, double>::type;
  constexpr int KB = MIXED ? 16 : 8;
  __shared__ double lds[NW];
  __shared__ int item_s;
  __shared__ VT lp[NW * KB * 64], lq[NW * KB * 64];
  double *work = a.work + (long long)blockIdx.x * a.stride;
  int q = blockIdx.x % kQueues, tried = 0;  // this XCD's queue first
  for (;;) {
    if (threadIdx.x == 0) item_s = next_item(a, q, tried);
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(item_s);
    __syncthreads();
    if (item < 0) break;
    const unsigned long long t_start = realtime();
    const int sidx = __builtin_amdgcn_readfirstlane(a.items[item].x);
    const int rhs = __builtin_amdgcn_readfirstlane(a.items[item].y);
    const StripView S = load_uniform(&a.sys[sidx].S);
    const int npad = load_uniform(&a.sys[sidx].npad);
    const double *b = load_uniform(&a.sys[sidx].b) + (long long)rhs * npad;
    double *x = load_uniform(&a.sys[sidx].x) + (long long)rhs * npad;
    double *part = work + 3 * (size_t)a.npad_max;
    ItemState st;
    double s2 = 0.0;
    for (int i = threadIdx.x; i < S.nrows; i += 64 * NW) s2 += b[i] * b[i];
    st.bb = block_sum(s2, lds);
    st.stop2 = a.tol2 * st.bb;
    if (st.bb != 0.0) {
      ItemEnd end;
      if (S.nstrips <= NW * KB)
        end = item_on_chip<NW, KB, VT>(a, S, b, x, lp, lq, part, lds, st);
      else
        end = item_in_memory<NW, VT>(a, S, b, x, work, npad, part, lds, st);
      if (MIXED && end == kItemNeeds64) {
        __syncthreads();
        ++st.refresh;
        (void)item_in_memory<NW, double>(a, S, b, x, work, npad, part, lds, st);
      }
    }
    __syncthreads();
    // FP64 relative residual of the result
    double fv = 0.0;
    block_product<NW>(S, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63, MemVec<double>{x}, false, part,
                      [&](int, int i, double ax, double) {
                        const double d = b[i] - ax;
                        fv += d * d;
                      });
    const double fin = block_sum(fv, lds);
    if (threadIdx.x == 0) {
      a.iters[item] = st.it;
      a.relres[item] = st.bb > 0.0 ? sqrt(fin / st.bb) : sqrt(fin);
      a.tstamp[2 * item] = t_start;
      a.tstamp[2 * item + 1] = realtime();
    }
    __syncthreads();
  }
}

const void *batch_strip_kernel(int waves, bool mixed) {
  switch (waves) {
    case 4: return mixed ? (const void *)k_batch_strip<4, true> : (const void *)k_batch_strip<4, false>;
    case 8: return mixed ? (const void *)k_batch_strip<8, true> : (const void *)k_batch_strip<8, false>;
    default: return mixed ? (const void *)k_batch_strip<16, true> : (const void *)k_batch_strip<16, false>;
  }
}

}  // namespace mf
