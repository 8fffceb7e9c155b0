// mf_strip_solve.hip -- persistent CG and BiCGSTAB over row strips, their
// vectors on chip.
//
// One cooperative launch runs the whole solve, as in mf_solve.hip, on the row
// strips of the handle (mf_strips.h): a wave owns up to kMaxWaveStrips strips,
// 64 rows each, one row per lane.  Only the vectors that a product gathers
// (CG: r) are in memory.  The search direction p, s = A p and the iterate x of the
// wave's rows stay in the lanes' registers for the whole solve, and w = A r
// and the own entries of r pass from the product to the update through the
// wave's part of the LDS, so an iteration reads the matrix and r and writes r
// (FP64: 16 bytes a row besides the matrix, instead of 80).  x goes to memory
// when the residual is recomputed, and at the end.
//
// Arithmetic: sums and scalars FP64.  Under a mixed policy r, p and s are
// rounded to FP32 where the tile solver stores them in FP32, and the strips
// multiply the FP32 payload (in FP64 arithmetic; packed strips hold it
// exactly).  A wave whose learned levels include FP64 runs its strips at FP64.
#include <cmath>
#include <type_traits>

#include "mf_strip_solve.h"

namespace mf {

namespace {

__device__ __forceinline__ int solver_wave() {
  const int G = gridDim.x;
  const int lb = (G & 7) ? (int)blockIdx.x : (int)(blockIdx.x & 7) * (G >> 3) + (int)(blockIdx.x >> 3);
  return __builtin_amdgcn_readfirstlane(lb * kWavesPerBlock + (int)(threadIdx.x >> 6));
}

// Store that writes through the XCD's L2 (see mf_solve.hip).
template <typename T>
__device__ __forceinline__ void wt(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double sum16(double v) {
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// The wave's strips s0 + k * step, k < n.
struct StripWave {
  int s0, step, n, lane;
};

// Sum of the pieces of lane's long row, posted by the waves that hold them
// (values tagged with the product's ordinal, as in grid_sum_values; waits are
// bounded).
// 2 D pieces are awaited at a time: one by one, a row of 32 pieces cost 32
// trips through memory (200k-row power law: 30.6 us an iteration, now 28.0).
template <int N>
__device__ __forceinline__ double take_pieces(const StripSolveArgs &a, int h, unsigned tag) {
  const LongRow lr = a.S.lrow[h];
  double sum = 0.0;
  for (int j = 0; j < lr.n; j += N) {
    unsigned long long q[2 * N];
    unsigned spins = 0;
    for (;;) {
      bool ok = true;
#pragma unroll
      for (int u = 0; u < 2 * N; ++u) {
        // (past the last piece: the last again, not added)
        const int i = min(j + u / 2, lr.n - 1);
        q[u] = __hip_atomic_load(a.pmail + 2 * (size_t)(lr.first + i) + (u & 1), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int u = 0; u < 2 * N; ++u) ok = ok && (unsigned)(q[u] >> 32) == tag;
      if (ok || !spin_on(spins, a.gs)) break;
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (j + u < lr.n)
        sum += __builtin_bit_cast(double, (q[2 * u + 1] & 0xffffffffull) << 32 | (q[2 * u] & 0xffffffffull));
  }
  return sum;
}

// Pairs of entries in flight in a product.  Eight strips of FP64 vectors are 48
// (BiCGSTAB 64) of a lane's 128 registers: with four pairs in flight besides, 12 of them
// went to memory and back in every iteration (128^3, 25 MB).  CG with two 26.2 us an
// iteration, with four 29.2; random values 39.8 / 41.2, 21 entries a row 50.0 / 50.3.
// At four strips a wave the two are mixed (900k rows of 21 packed entries 27.8 /
// 26.0, 7 diagonals 13.9 / 14.1), and the mixed kernels lose (128^3 29.9 / 24.5).
template <int KS, bool MIXED>
constexpr int kDepth = KS == 8 && !MIXED ? 2 : 4;

// Products of the wave's pieces (posted for the rows' owners), then of its
// strips: w and (own_out) the rows' own entries of x to wl and rl (lane's slot of
// strip k at 64 k), and the sums of own^2, w * own and w^2.  Pieces never
// wait, and an owner waits only after its own pieces, so every wait ends.
template <bool EARLY, int D, typename XT>
__device__ __forceinline__ void strip_product(const StripSolveArgs &a, const StripWave &w, const XT *__restrict__ x,
                                              unsigned tag, bool v32, bool own_out, double *wl, double *rl,
                                              double (&g)[3]) {
  const StripView &S = a.S;
  g[0] = g[1] = g[2] = 0.0;
  if (S.npieces > 0) {
    const int wid = solver_wave();
    const int q1 = __builtin_amdgcn_readfirstlane(a.wave_piece[wid + 1]);
    for (int q = __builtin_amdgcn_readfirstlane(a.wave_piece[wid]); q < q1; ++q) {
      const int pc = __builtin_amdgcn_readfirstlane(a.piece_order[q]);
      const double v[1] = {piece_sum<D>(S, pc, w.lane, MemVec<XT>{x}, v32)};
      if (w.lane == 0) mbox_post<1>(a.pmail + 2 * (size_t)pc, tag, v);
    }
  }
  int o = w.lane - 64;
  strips_run<EARLY, D>(S, w.lane, MemVec<XT>{x}, v32, w.n, [&](int k) { return w.s0 + k * w.step; },
             [&](int s, const StripDesc &d, int, bool lng, double acc, double own) {
               if ((d.flags & kStripLong) && lng) acc += take_pieces<2 * D>(a, S.lane_long[64 * s + w.lane], tag);
               o += 64;
               wl[o] = acc;
               if (own_out) rl[o] = own;
               g[0] += own * own;
               g[1] += acc * own;
               g[2] += acc * acc;
             });
}

// Tiles [t0, t1) counted per level (wave-uniform).
__device__ __forceinline__ void count_levels(const uint8_t *prec, int t0, int t1, int lane, unsigned (&n)[5]) {
#pragma unroll
  for (int l = 0; l < 5; ++l) n[l] = 0;
  for (int t = t0; t < t1; t += kWave) {
    const int u = t + lane;
    const int p = u < t1 ? prec[u] : 255;
#pragma unroll
    for (int l = 0; l < 5; ++l) n[l] += (unsigned)__builtin_popcountll(__ballot(p == l));
  }
}

// The wave's strips, and the tiles whose levels it counts and infers: of
// unsorted strips, its share of the tiles that the block's strips hold (learned
// levels are inferred there, and a block with an FP64 tile multiplies FP64); of
// sorted ones, which no learned solve takes, an equal share of all.
// Unsorted strips go round the waves of their block, so that the block's waves
// gather from neighbouring rows at the same time (L1; FP64 64^3 9.5 us an iteration
// with contiguous strips, now 9.3; error bound 128^3 25.6 and 24.9).  Sorted
// ones stay contiguous: a window's longest come first.
__device__ __forceinline__ void wave_share(const StripSolveArgs &a, int wid, int lane, StripWave &W, int &t0, int &t1) {
  const int nw = gridDim.x * kWavesPerBlock, wv = wid % kWavesPerBlock;
  W.lane = lane;
  if (a.S.rowmap) {
    W.s0 = (int)((long long)a.S.nstrips * wid / nw);
    W.step = 1;
    W.n = (int)((long long)a.S.nstrips * (wid + 1) / nw) - W.s0;
    t0 = (int)((long long)a.A.tilenum * wid / nw);
    t1 = (int)((long long)a.A.tilenum * (wid + 1) / nw);
  } else {
    const int b = wid / kWavesPerBlock, G = gridDim.x;
    const int b0 = (int)((long long)a.S.nstrips * b / G), b1 = (int)((long long)a.S.nstrips * (b + 1) / G);
    W.s0 = b0 + wv;
    W.step = kWavesPerBlock;
    W.n = max(b1 - W.s0 + kWavesPerBlock - 1, 0) / kWavesPerBlock;
    // (a strip is four tile-rows)
    const int u0 = load_uniform(a.A.tile_ptr + min(4 * b0, a.A.tilem));
    const int u1 = load_uniform(a.A.tile_ptr + min(4 * b1, a.A.tilem));
    t0 = u0 + (int)((long long)(u1 - u0) * wv / kWavesPerBlock);
    t1 = u0 + (int)((long long)(u1 - u0) * (wv + 1) / kWavesPerBlock);
  }
}

// Row of the lane in strip s0 + k.  The lane is hidden from the optimizer,
// which would otherwise keep every strip's row and row-map address in
// registers for the whole solve.
__device__ __forceinline__ int wave_row(const StripSolveArgs &a, const StripWave &W, int k) {
  int l = W.lane;
  asm("" : "+v"(l));
  bool lng;
  return strip_row(a.S, W.s0 + k * W.step, l, lng);
}

__device__ __forceinline__ void add_hist(unsigned long long c, unsigned long long *h, int lane) {
  if (lane == 0 && c) atomicAdd(h, c);
}

}  // namespace

// Inference context for a multiplied vector of squared norm v2.
__device__ __forceinline__ InferCtx infer_ctx(const StripSolveArgs &a, double v2, double rr, double bb) {
  InferCtx c;
  c.w = a.mlp;
  c.feat16 = a.feat16;
  c.seg2 = a.seg2;
  c.prec_out = a.prec_rw;
  c.seg_scale = v2 > 0.0 ? (float)(sqrt((double)a.nseg) / sqrt(v2)) : 0.0f;
  c.progress = (float)(log10(fmax(bb > 0.0 ? sqrt(rr / bb) : 1.0, 1e-16)) / 16.0);
  return c;
}

// Learned levels of tiles [t0, t1) from the installed network.  Out of line:
// it runs once per check interval, and inlined its 36 operand registers were
// spilled around every product.
__device__ __noinline__ void infer_levels(const int *tile_col, InferCtx c, int t0, int t1, int lane) {
  TileView A;
  A.tile_col = tile_col;
  wave_infer_tiles<false>(A, c, t0, t1, lane);
}

// Chronopoulos-Gear CG: w = A r with gamma = r.r and delta = w.r, one fused
// grid sum, then p = r + beta p, s = w + beta s, x += alpha p, r -= alpha s and
// a grid sync (the exits, refreshes and fallback of k_cg; a mixed solve that
// needs FP64 ends, and the host starts an FP64 one from its x).
//
// Measured on MI355X, us per iteration, FP64 / error bound (streamed tiles with
// the vectors in memory before): 7-point 128^3 26.2 / 24.5 (54.0 / 45.0), of
// which the update's stores 6.5 and the two synchronisations 7.6;
// 117 x 89 x 86 14.1 / 16.0 (30.0 / 29.4); 64^3 9.3 / 10.7 (16.7 / 18.7), of
// which synchronisation 6; 5-point 64^2 5.1 / 6.4 (10.8 / 13.3); 200k-row power
// law 27.5 / 26.4 (97 / 107).  The 128^3 product moves 40 MB.
//
// Each round of the
// loop is one product: of x for a residual (kRes), of r for an iteration
// (kIter) or of p for s after a refresh (kDir).
template <int KS, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_cg_strip(StripSolveArgs a) {
  using VT = typename std::conditional<MIXED, float, double>::type;
  enum Round { kRes, kIter, kDir };
  __shared__ double lds[kMaxGridSum * kWavesPerBlock];
  __shared__ double lw[kWavesPerBlock][KS * 64];  // A times the vector, of the wave's rows
  __shared__ double lr[kWavesPerBlock][KS * 64];  // the vector's own entries
  const int wid = solver_wave();
  double *wl = lw[threadIdx.x >> 6], *rl = lr[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  StripWave W;
  int t0, t1;
  wave_share(a, wid, lane, W, t0, t1);
  auto row_of = [&](int k) { return wave_row(a, W, k); };
  unsigned epoch = 0, tag = 0;
  int slot = 0, lds_i = 0;
  VT p[KS], s[KS];
  double x[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    p[k] = s[k] = VT(0);
    x[k] = 0.0;
    if (k < W.n) {
      const int row = row_of(k);
      if (row >= 0) x[k] = a.x[row];
    }
  }
  const bool learned = MIXED && a.mlp != nullptr;
  double rr = 0.0, bb = 0.0, stop2 = 0.0, rr_ref = 0.0, gamma_old = 1.0, alpha_old = 1.0;
  int it = 0, it_ref = 0, refresh = -1, status = 0;
  bool first = true;      // the next step starts a new direction
  bool fell = false;      // mixed: stopped for the FP64 solver to go on
  bool infer = learned;   // new levels in the next product
  bool full64 = false;    // FP64 payload under FP32 vectors (learned FP64 levels)
  bool end = false;       // this residual is the last one, for the report
  unsigned nlev[5] = {0, 0, 0, 0, 0};  // the wave's tiles per level
  unsigned long long hist[5] = {0, 0, 0, 0, 0};
  if (MIXED && !learned) count_levels(a.A.prec, t0, t1, lane, nlev);

  Round round = kRes;
  for (;;) {
    double gd3[3];
    ++tag;
    if (MIXED && round == kIter) {
      if (infer) {
        infer_levels(a.A.tile_col, infer_ctx(a, rr, rr, bb), t0, t1, lane);
        count_levels(a.prec_rw, t0, t1, lane, nlev);
        full64 = __syncthreads_or(nlev[0] > 0);  // (the block's strips hold these tiles)
        infer = false;
      }
      strip_product<!MIXED, kDepth<KS, MIXED>>(a, W, (const float *)a.r32, tag, !full64, true, wl, rl, gd3);
    } else {
      const double *v = round == kRes ? a.x : round == kIter ? a.r : a.p;
      strip_product<!MIXED, kDepth<KS, MIXED>>(a, W, v, tag, false, true, wl, rl, gd3);
    }
    if (round == kRes) {
      // r = b - A x of the wave's rows (stored unless it is the last)
      double tr[2] = {0.0, 0.0};
      for (int k = 0; k < W.n; ++k) {
        const int row = row_of(k);
        if (row >= 0) {
          const double bv = a.b[row];
          double rv = bv - wl[64 * k + lane];
          if (MIXED && !end) {
            const float rf = (float)rv;
            a.r32[row] = rf;
            rv = rf;
          } else if (!end) {
            a.r[row] = rv;
          }
          tr[0] += rv * rv;
          tr[1] += bv * bv;
          if (learned && refresh < 0) {
            // segment norms of r0 for the first inference
            const double d2 = sum16(rv * rv);
            if ((lane & 15) == 0) a.seg2[row >> 4] = (float)d2;
          }
        }
      }
      grid_sum<2>(tr, a.partials, a.gs, epoch, slot, lds, &lds_i);
      if (end) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
          a.stats[kStIters] = it;
          a.stats[kStRefresh] = refresh;
          a.stats[kStFallback] = fell;
          a.stats[kStRecursive] = rr;
          a.stats[kStTrue] = tr[0];
          a.stats[kStBB] = bb;
          a.stats[kStStatus] = status;
        }
        break;
      }
      ++refresh;
      if (refresh == 0) {  // the initial residual
        bb = tr[1];
        stop2 = uniform_double(a.tol2 * bb);
        rr = rr_ref = tr[0];
        if (bb == 0.0 || (a.fixed_iters <= 0 && rr <= stop2)) {
          end = true;
        } else {
          round = kIter;
        }
        continue;
      }
      it_ref = it;
      // A recursive residual far below the true one leaves beta meaningless,
      // and so does one that met the tolerance while the true one did not:
      // restart the search direction from the recomputed residual.
      if (tr[0] > 4.0 * rr || (rr <= stop2 && tr[0] > stop2)) first = true;
      rr = tr[0];
      if (tr[0] <= stop2) {
        end = true;
        continue;
      }
      if (it >= a.maxiter) {
        status = MF_NOT_CONVERGED;
        end = true;
        continue;
      }
      if (MIXED && (tr[0] > 0.25 * rr_ref || refresh > a.max_refresh)) {
        // stagnation: x is the start of an FP64 solve
        fell = end = true;
        continue;
      }
      rr_ref = rr;
      if (first) {
        round = kIter;
        grid_sync(a.gs, epoch, &lds_i);
      } else {
        // s = A p in FP64 so that s and the new r stay consistent
        round = kDir;
#pragma unroll
        for (int k = 0; k < KS; ++k)
          if (k < W.n) {
            const int row = row_of(k);
            if (row >= 0) wt(a.p + row, (double)p[k]);
          }
        grid_sync(a.gs, epoch, &lds_i);
      }
      continue;
    }
    if (round == kDir) {
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) s[k] = (VT)wl[64 * k + lane];
      round = kIter;
      // (a wave that went on would post the next product's piece sums over
      // these)
      grid_sync(a.gs, epoch, &lds_i);
      continue;
    }
    if (MIXED) {
#pragma unroll
      for (int l = 0; l < 5; ++l) hist[l] += nlev[l];
    }
    double gd[2] = {gd3[0], gd3[1]};
    grid_sum_values<2>(gd, a.mbox, a.gs, epoch, lds);
    const double gamma = gd[0], delta = gd[1];
    rr = gamma;
    bool pending = false;  // recompute the FP64 residual before the step
    if (a.fixed_iters <= 0) {
      pending = gamma <= stop2 || (MIXED &&
                                   (gamma <= a.ratio2 * rr_ref || it - it_ref >= a.refresh_every));
      if (!pending && it >= a.maxiter) {
        status = MF_NOT_CONVERGED;
        end = true;
      }
    }
    double beta = 0.0, alpha = gamma / delta;
    if (!first) {
      beta = gamma / gamma_old;
      alpha = gamma / (delta - beta * gamma / alpha_old);
    }
    if (!pending && !end && (!isfinite(alpha) || alpha == 0.0 || (MIXED && !(alpha > 0.0)))) {
      // (a low-precision operator that lost definiteness: FP64 goes on)
      if (MIXED) fell = true;
      else status = MF_ERR_BREAKDOWN;
      end = true;
    }
    const bool step = !pending && !end;
    // p = r + beta p, x += alpha p: needed by no other wave, so done while the
    // arrivals of the other blocks are awaited
    auto update_px = [&] {
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) {
          p[k] = (VT)(rl[64 * k + lane] + beta * (double)p[k]);
          x[k] += alpha * (double)p[k];
        }
    };
    if (step) {
      first = false;
      alpha = uniform_double(alpha);
      beta = uniform_double(beta);
      gamma_old = gamma;
      alpha_old = alpha;
      ++it;
      const bool lupd = learned && (it % a.check_interval) == 0;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if (k < W.n) {
          const int row = row_of(k);
          // (mixed: w, p, s and r rounded to FP32 as the tile solver stores them)
          s[k] = (VT)((double)(VT)wl[64 * k + lane] + beta * (double)s[k]);
          const VT rn = (VT)(rl[64 * k + lane] - alpha * (double)s[k]);
          if (row >= 0) wt((MIXED ? (VT *)a.r32 : (VT *)a.r) + row, rn);
          if (MIXED && lupd) {
            const double d = sum16(row >= 0 ? (double)rn * (double)rn : 0.0);
            if ((lane & 15) == 0 && row >= 0) wt(a.seg2 + (row >> 4), (float)d);
          }
        }
      }
      infer = lupd;
      end = a.fixed_iters > 0 && it >= a.fixed_iters;
    }
    if (pending || end) {
      // x to memory, for the residual
      if (step) update_px();
      round = kRes;
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) {
          const int row = row_of(k);
          if (row >= 0) wt(a.x + row, x[k]);
        }
    }
    grid_arrive<false>(a.gs, epoch);
    if (step && !end) update_px();
    grid_wait(a.gs, epoch);
  }
  if (MIXED) {
#pragma unroll
    for (int l = 0; l < 5; ++l) add_hist(hist[l], a.hist + l, lane);
  }
}


// BiCGSTAB (van der Vorst) over row strips, with the scalars, exits, restarts
// and refreshes of k_bicgstab.  Gathered, and so in memory: p and s.  Of the
// wave's rows, x, r^, v and r (s between the two products) are in registers,
// p's own entries in rl from its product on, and t = A s in wl.  Each round is
// one product: of x (kRes), p or s.  A mixed solve that breaks down or
// stagnates ends, and the host starts an FP64 one from its x.
//
// Measured on MI355X, convection-diffusion 100^3, us per iteration: FP64 32.4,
// error bound 34.0 (tiles with the vectors in memory: 67.8 and 59.7): two
// products of about 7 us, three sums and two barriers of 15 us together.
constexpr int kStripRestarts = 8;

template <int KS, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_bicgstab_strip(StripSolveArgs a) {
  using VT = typename std::conditional<MIXED, float, double>::type;
  enum Round { kRes, kP, kS };
  __shared__ double lds[kMaxGridSum * kWavesPerBlock];
  __shared__ double lw[kWavesPerBlock][KS * 64];
  __shared__ double lr[kWavesPerBlock][KS * 64];
  const int wid = solver_wave();
  double *wl = lw[threadIdx.x >> 6], *rl = lr[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  StripWave W;
  int t0, t1;
  wave_share(a, wid, lane, W, t0, t1);
  auto row_of = [&](int k) { return wave_row(a, W, k); };
  VT *const gp = MIXED ? (VT *)a.p32 : (VT *)a.p, *const gs_ = MIXED ? (VT *)a.r32 : (VT *)a.r;
  unsigned epoch = 0, tag = 0;
  int slot = 0, lds_i = 0;
  VT rs[KS], rh[KS], v[KS];
  double x[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    rs[k] = rh[k] = v[k] = VT(0);
    x[k] = 0.0;
    if (k < W.n) {
      const int row = row_of(k);
      if (row >= 0) x[k] = a.x[row];
    }
  }
  const bool learned = MIXED && a.mlp != nullptr;
  double rho = 0.0, rr = 0.0, rho_new = 0.0, rr_new = 0.0, bb = 0.0, stop2 = 0.0, rr_ref = 0.0, pp_last = 0.0;
  double alpha = 0.0, omega = 0.0;
  int it = 0, it_ref = 0, refresh = -1, restarts = 0, status = 0;
  bool fresh = true;     // this residual starts r, r^ and p anew
  bool infer = learned, full64 = false, fell = false, end = false;
  unsigned nlev[5] = {0, 0, 0, 0, 0};
  unsigned long long hist[5] = {0, 0, 0, 0, 0};
  if (MIXED && !learned) count_levels(a.A.prec, t0, t1, lane, nlev);
  // x to memory and a grid barrier, before a residual
  auto sync_x = [&] {
#pragma unroll
    for (int k = 0; k < KS; ++k)
      if (k < W.n) {
        const int row = row_of(k);
        if (row >= 0) wt(a.x + row, x[k]);
      }
    grid_arrive<false>(a.gs, epoch);
    grid_wait(a.gs, epoch);
  };

  Round round = kRes;
  for (;;) {
    double gd[3];
    ++tag;
    if (MIXED && round != kRes) {
      if (round == kP && infer) {
        infer_levels(a.A.tile_col, infer_ctx(a, pp_last, rr, bb), t0, t1, lane);
        count_levels(a.prec_rw, t0, t1, lane, nlev);
        full64 = __syncthreads_or(nlev[0] > 0);  // (the block's strips hold these tiles)
        infer = false;
      }
      strip_product<false, kDepth<KS, MIXED>>(a, W, (const float *)(round == kP ? gp : gs_), tag, !full64, round == kP, wl, rl, gd);
    } else {
      const double *u = round == kRes ? a.x : (const double *)(round == kP ? gp : gs_);
      strip_product<false, kDepth<KS, MIXED>>(a, W, u, tag, false, round == kP, wl, rl, gd);
    }
    bool step = false;  // go on to p = r + beta (p - omega v)
    bool restart = false;
    if (round == kRes) {
      double tr[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) {
          const int row = row_of(k);
          if (row >= 0) {
            const double bv = a.b[row];
            double rv = bv - wl[64 * k + lane];
            if (!end) {
              rs[k] = (VT)rv;
              rv = (double)rs[k];
              if (fresh) {
                rh[k] = rs[k];
                wt(gp + row, rs[k]);
              }
            }
            tr[0] += rv * rv;
            tr[1] += rv * (double)rh[k];
            tr[2] += bv * bv;
            if (MIXED && learned && refresh < 0) {
              // segment norms of p = r0 for the first inference
              const double d2 = sum16(rv * rv);
              if ((lane & 15) == 0) wt(a.seg2 + (row >> 4), (float)d2);
            }
          }
        }
      grid_sum<3>(tr, a.partials, a.gs, epoch, slot, lds, &lds_i);
      if (end) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
          a.stats[kStIters] = it;
          a.stats[kStRefresh] = refresh;
          a.stats[kStFallback] = fell;
          a.stats[kStRecursive] = rr;
          a.stats[kStTrue] = tr[0];
          a.stats[kStBB] = bb;
          a.stats[kStStatus] = status;
        }
        break;
      }
      ++refresh;
      it_ref = it;
      if (fresh) {
        if (refresh == 0) {
          bb = tr[2];
          stop2 = uniform_double(a.tol2 * bb);
          pp_last = tr[0];
        }
        rr = rho = rr_ref = tr[0];
        fresh = false;
        if (bb == 0.0 || ((a.fixed_iters <= 0 || refresh > 0) && rr <= stop2)) {
          end = true;
          continue;
        }
        ++it;
        round = kP;
        continue;
      }
      if (tr[0] <= stop2) {
        rr = tr[0];
        end = true;
        continue;
      }
      if (MIXED && it < a.maxiter && (tr[0] > 0.25 * rr_ref || refresh > a.max_refresh)) {
        rr = tr[0];
        fell = end = true;
        continue;
      }
      // A recursive residual far below the true one makes beta meaningless.
      restart = tr[0] > 4.0 * rr_new;
      rr_new = rr_ref = tr[0];
      rho_new = tr[1];
      step = true;
    } else if (round == kP) {
      // v = A p, alpha = rho / (v . r^), s = r - alpha v
      double vr[1] = {0.0};
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) {
          const double vv = wl[64 * k + lane];
          vr[0] += vv * (double)rh[k];
          v[k] = (VT)vv;
        }
      if (MIXED) {
#pragma unroll
        for (int l = 0; l < 5; ++l) hist[l] += 2 * nlev[l];
      }
      grid_sum_values<1>(vr, a.mbox, a.gs, epoch, lds);
      if (!(vr[0] != 0.0) || !isfinite(vr[0])) {
        if (MIXED) fell = end = true;
        restart = true;
      } else {
        alpha = uniform_double(rho / vr[0]);
#pragma unroll
        for (int k = 0; k < KS; ++k)
          if (k < W.n) {
            const int row = row_of(k);
            rs[k] = (VT)((double)rs[k] - alpha * (double)v[k]);
            if (row >= 0) wt(gs_ + row, rs[k]);
          }
        grid_arrive<false>(a.gs, epoch);
        grid_wait(a.gs, epoch);
        round = kS;
        continue;
      }
    } else {
      // t = A s, omega = t.s / t.t, x += alpha p + omega s, r = s - omega t
      double tw[2] = {gd[1], gd[2]};
      grid_sum_values<2>(tw, a.mbox, a.gs, epoch, lds);
      omega = uniform_double(tw[1] != 0.0 && isfinite(tw[1]) ? tw[0] / tw[1] : 0.0);
      double nw[2] = {0.0, 0.0};
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < W.n) {
          const double sv = (double)rs[k];
          x[k] += alpha * rl[64 * k + lane] + omega * sv;
          rs[k] = (VT)(sv - omega * wl[64 * k + lane]);
          nw[0] += (double)rs[k] * (double)rh[k];
          nw[1] += (double)rs[k] * (double)rs[k];
        }
      grid_sum_values<2>(nw, a.mbox, a.gs, epoch, lds);
      rho_new = nw[0];
      rr_new = nw[1];
      if (a.fixed_iters > 0) {
        if (it >= a.fixed_iters) {
          rr = rr_new;
          end = true;
        } else {
          step = true;
        }
      } else if (rr_new <= stop2 || omega == 0.0 || !isfinite(rr_new) ||
                 (MIXED && (rr_new <= a.ratio2 * rr_ref || it - it_ref >= a.refresh_every))) {
        // the FP64 residual first (p, v and the scalars of this step are kept)
        round = kRes;
        sync_x();
        continue;
      } else {
        step = true;
      }
    }
    if (step && !restart && a.fixed_iters <= 0) {
      if (it >= a.maxiter) {
        rr = rr_new;
        status = MF_NOT_CONVERGED;
        end = true;
      } else if (omega == 0.0 || rho == 0.0 || rho_new == 0.0 || !isfinite(rho_new)) {
        restart = true;
      }
    } else if (step && restart && it >= a.maxiter) {
      rr = rr_new;
      status = MF_NOT_CONVERGED;
      end = true;
    }
    if (restart && !end && ++restarts > kStripRestarts) {
      status = MF_ERR_BREAKDOWN;
      end = true;
    }
    if (restart || end) {
      round = kRes;
      fresh = true;
      sync_x();
      continue;
    }
    const double beta = uniform_double((rho_new / rho) * (alpha / omega));
    rho = rho_new;
    rr = rr_new;
    const bool lupd = learned && (it % a.check_interval) == 0;
    double pp[1] = {0.0};
#pragma unroll
    for (int k = 0; k < KS; ++k)
      if (k < W.n) {
        const int row = row_of(k);
        const VT pv = (VT)((double)rs[k] + beta * (rl[64 * k + lane] - omega * (double)v[k]));
        if (row >= 0) wt(gp + row, pv);
        if (MIXED && lupd) {
          const double d = row >= 0 ? (double)pv * (double)pv : 0.0, d2 = sum16(d);
          pp[0] += d;
          if ((lane & 15) == 0 && row >= 0) wt(a.seg2 + (row >> 4), (float)d2);
        }
      }
    if (lupd) {
      grid_sum<1>(pp, a.partials, a.gs, epoch, slot, lds, &lds_i);
      pp_last = pp[0];
      infer = true;
    } else {
      grid_arrive<false>(a.gs, epoch);
      grid_wait(a.gs, epoch);
    }
    ++it;
    round = kP;
  }
  if (MIXED) {
#pragma unroll
    for (int l = 0; l < 5; ++l) add_hist(hist[l], a.hist + l, lane);
  }
}

template <int KS>
static const void *strip_kernel(bool bicg, bool mixed) {
  if (bicg) return mixed ? (const void *)k_bicgstab_strip<KS, true> : (const void *)k_bicgstab_strip<KS, false>;
  return mixed ? (const void *)k_cg_strip<KS, true> : (const void *)k_cg_strip<KS, false>;
}

const void *strip_solve_kernel(int strips, bool bicg, bool mixed) {
  if (strips <= 1) return strip_kernel<1>(bicg, mixed);
  if (strips <= 2) return strip_kernel<2>(bicg, mixed);
  if (strips <= 4) return strip_kernel<4>(bicg, mixed);
  return strip_kernel<8>(bicg, mixed);
}

}  // namespace mf
