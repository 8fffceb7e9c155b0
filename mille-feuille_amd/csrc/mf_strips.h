// mf_strips.h -- row strips: the device layout with one matrix row per lane,
// and its product.
//
// A strip is 64 rows, one per lane of a wave.  Entry k of all 64 rows is
// stored together, two entries at a time (lane l's entries 2k and 2k+1 at
// 128 k + 2 l), so a wave reads its strip with coalesced 8- or 16-byte loads,
// keeps every row sum in a register and needs neither LDS nor atomics; in a
// banded matrix the lanes' gathers of x fall in consecutive addresses too.
// Rows are padded to the longest of their strip.  Where consecutive rows
// differ too much for that (see build_strips), the rows of each window of
// kStripWin strips are sorted by length first, and rows longer than
// kLongRow entries go to pieces: a piece has the layout of a strip whose 64
// lanes all hold entries of one row.
//
// Four classes (where every row of a strip has a diagonal entry, the strip's
// diagonals are stored apart, the lead: lead64, lead32):
//   diagonal (kStripDiag): every entry but the lead lies on a diagonal that has
//     one value in the strip (constant-coefficient stencils in any numbering
//     that keeps them banded): per diagonal a mask of rows, the offset and the
//     FP64 value, read by scalar loads.  No bytes per entry, and fewer instructions
//     than a packed one.  Measured on MI355X against the packed class, hot / cold us:
//     128^3 7-point product 17.4 / 36.5, now 16.1 / 30.6; 117 x 89 x 86 9.3 / 19.7,
//     now 6.8 / 15.7; CG with the error bound 128^3 28.4 us an iteration, now 24.6.
//   packed (kStripPacked): every entry but the lead in one 32-bit word, column
//     field << 8 | (q + 128) with value q * scale, |q| <= 127 and scale a power
//     of two common to the strip.  Used only where that holds every value
//     exactly (graph Laplacians, constant-coefficient stencils), so the
//     products are those of the FP64 values; 4 bytes an entry instead of 9.
//   near (kStripNear): FP64 and FP32 values and 16-bit column fields.
//   full (kStripFull): FP64 and FP32 values and 32-bit columns.
// Padding gathers an entry of x that exists, and its product is replaced by 0,
// so an infinity or NaN in x reaches exactly the rows that have an entry in its column.
#pragma once

#include <type_traits>

#include "mf_device.h"

namespace mf {

struct StripView {
  const StripDesc *desc;   // strips, then pieces
  const uint32_t *words;   // packed entries
  const double *vv;        // full entries: FP64 values, FP32 values, columns
  const float *vf;
  const int *vc;           // (-1: padding)
  const uint16_t *vh;      // near columns (0: padding)
  const DiagSlot *dslot;   // diagonals
  const double *lead64;    // diagonal of strip lane 64 s + lane
  const float *lead32;
  const int *rowmap;       // row of each strip lane (sorted layouts; -1: none), else null
  const int *lane_long;    // long row of each strip lane (layouts with pieces), else null
  const LongRow *lrow;     // nlong
  const int *piece_long;   // long row of each piece
  int nstrips, npieces, nlong, nmulti, nrows;
  int leads;  // half of the strips or more have a lead
};

inline StripView strip_view_of(const mf_tiled *t) {
  const StripLayout &s = t->strips;
  return StripView{s.desc, s.words, s.vv, s.vf, s.vc, s.vh, s.dslot, s.lead64, s.lead32, s.rowmap,
                   s.lane_long, s.lrow, s.piece_long, s.nstrips, s.npieces, s.nlong, s.nmulti,
                   16 * t->tilem, s.leads};
}

// Row of the lane's strip slot: its row, or -1; `lng` is set for a row whose
// other entries are in pieces.
__device__ __forceinline__ int strip_row(const StripView &S, int s, int lane, bool &lng) {
  lng = false;
  if (!S.rowmap) {
    const int r = 64 * s + lane;
    return r < S.nrows ? r : -1;
  }
  const int r = S.rowmap[64 * s + lane];
  if (r < 0) return -1;
  lng = (r & kLongBit) != 0;
  return r & (kLongBit - 1);
}

// *p for a wave-uniform p by scalar loads: data that does not change while
// kernels run, which the constant address space tells the compiler.
template <typename T>
__device__ __forceinline__ T load_uniform(const T *p) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  typedef const __attribute__((address_space(4))) uint32_t *ConstPtr;
  const ConstPtr q = (ConstPtr)(uintptr_t)p;
  struct Raw { uint32_t w[sizeof(T) / 4]; } u;
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 4); ++k) u.w[k] = q[k];
  return __builtin_bit_cast(T, u);
}

// The vector that a strip multiplies: in memory, or in the block's LDS.
// rebase(d).get(i) is entry i + d.
template <typename T>
struct MemVec {
  typedef T value;
  const T *p;
  __device__ __forceinline__ MemVec rebase(ptrdiff_t d) const { return MemVec{p + d}; }
  __device__ __forceinline__ T get(uint32_t i) const { return ld_at<T>(p, i * (uint32_t)sizeof(T)); }
};

template <typename T>
struct LdsVec {
  typedef T value;
  const T *p;
  int off = 0;
  __device__ __forceinline__ LdsVec rebase(ptrdiff_t d) const { return LdsVec{p, off + (int)d}; }
  __device__ __forceinline__ T get(uint32_t i) const { return p[(int)i + off]; }
};

// The lane's N word pairs at byte offset vo of the strip's words.
template <int N>
__device__ __forceinline__ void strip_load_words(const uint32_t *__restrict__ w, uint32_t vo, uint2 (&r)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) r[i] = ld_at<uint2>(w, vo + 512u * i);
}

// Adds the products of N loaded word pairs to acc.  xb starts 2^23 entries
// before the strip's base row (an address only: the packed column field is
// biased by 2^23).
template <int N, class X>
__device__ __forceinline__ double strip_packed(const uint2 (&w)[N], const X &xb, float sc, double acc) {
  typename X::value g[2 * N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    g[2 * i] = xb.get(w[i].x >> 8);
    g[2 * i + 1] = xb.get(w[i].y >> 8);
  }
#pragma unroll
  for (int i = 0; i < 2 * N; ++i) {
    const uint32_t u = (i & 1 ? w[i / 2].y : w[i / 2].x) & 255u;
    // (u - 128) * scale, exact in FP32
    const float a = __builtin_fmaf((float)u, sc, -128.0f * sc);
    acc = __builtin_fma((double)a, u ? (double)g[i] : 0.0, acc);
  }
  return acc;
}

// The last pairs of a packed strip: four loaded ones and the np - k (< 4) after them.
template <class X>
__device__ __forceinline__ double strip_packed_rest(const uint32_t *__restrict__ w, uint32_t vo, int k, int np,
                                                    const uint2 (&a)[4], const X &xb, float sc, double acc) {
  if (np - k >= 2) {
    uint2 c[2];
    strip_load_words(w, vo + 512u * k, c);
    acc = strip_packed(a, xb, sc, acc);
    acc = strip_packed(c, xb, sc, acc);
    k += 2;
  } else {
    acc = strip_packed(a, xb, sc, acc);
  }
  if (np > k) {
    uint2 c[1];
    strip_load_words(w, vo + 512u * k, c);
    acc = strip_packed(c, xb, sc, acc);
  }
  return acc;
}

// N value / column pairs of a full or near strip from the lane's entry e;
// VT double or float.  Near columns: xb starts 2^15 entries before the base.
template <bool NEAR, int N, typename VT, class X>
__device__ __forceinline__ double strip_full(const VT *__restrict__ v, const void *__restrict__ c, uint32_t e,
                                             const X &xb, double acc) {
  VT a[2 * N];
  uint32_t j[2 * N];
  typename X::value g[2 * N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    struct alignas(2 * sizeof(VT)) Pair { VT x, y; };
    const Pair p = ld_at<Pair>(v, (e + 128u * i) * (uint32_t)sizeof(VT));
    a[2 * i] = p.x;
    a[2 * i + 1] = p.y;
    if constexpr (NEAR) {
      const uint32_t q = ld_at<uint32_t>(c, (e + 128u * i) * 2u);
      j[2 * i] = q & 0xffffu;
      j[2 * i + 1] = q >> 16;
    } else {
      const uint2 q = ld_at<uint2>(c, (e + 128u * i) * 4u);
      j[2 * i] = q.x;
      j[2 * i + 1] = q.y;
    }
  }
  // (padding gathers an entry that exists: the base row's, or x[0])
  auto pad = [](uint32_t q) { return NEAR ? q == 0u : (int)q < 0; };
#pragma unroll
  for (int i = 0; i < 2 * N; ++i)
    g[i] = xb.get(pad(j[i]) ? (NEAR ? 1u << 15 : 0u) : j[i]);
#pragma unroll
  for (int i = 0; i < 2 * N; ++i) acc = __builtin_fma((double)a[i], pad(j[i]) ? 0.0 : (double)g[i], acc);
  return acc;
}

template <bool NEAR, int D, typename VT, class X>
__device__ __forceinline__ double strip_full_sum(const VT *__restrict__ v, const void *__restrict__ c, int np,
                                                 int lane, const X &xb, double acc) {
  const uint32_t e = 2u * lane;
  int k = 0;
  for (; k + D <= np; k += D) acc = strip_full<NEAR, D>(v, c, e + 128u * k, xb, acc);
  const int rest = np - k;
  if constexpr (D > 3)
    if (rest == 3) return strip_full<NEAR, 3>(v, c, e + 128u * k, xb, acc);
  if (rest == 2) return strip_full<NEAR, 2>(v, c, e + 128u * k, xb, acc);
  if (rest == 1) return strip_full<NEAR, 1>(v, c, e + 128u * k, xb, acc);
  return acc;
}

// Sum of the lane's entries of a strip or piece (without the lead), added to
// acc.  X: the vector (MemVec or LdsVec); v32 (FP32 vectors only): full and
// near strips multiply the FP32 payload.  D: pairs in flight.  At four, packed
// strips of more than four pairs load
// the next four word pairs before the gathers of the current ones (two
// buffers in turn: a copy of words in flight would wait for them).
template <int D = 4, class X>
__device__ __forceinline__ double strip_sum(const StripView &S, const StripDesc &d, const X &x, int lane,
                                            double acc, bool v32 = false) {
  const int np = d.npair;
  if (d.cls == kStripPacked) {
    const uint32_t *w = S.words + (size_t)d.off * 128;
    const X xb = x.rebase((ptrdiff_t)d.base - (1 << 23));
    const uint32_t vo = 8u * lane;
    if (np <= 4) {
      if (np == 1) {
        uint2 a[1];
        strip_load_words(w, vo, a);
        return strip_packed(a, xb, d.scale, acc);
      }
      if (np == 2) {
        uint2 a[2];
        strip_load_words(w, vo, a);
        return strip_packed(a, xb, d.scale, acc);
      }
      if (np == 3) {
        uint2 a[3];
        strip_load_words(w, vo, a);
        return strip_packed(a, xb, d.scale, acc);
      }
      if (np == 4) {
        uint2 a[4];
        strip_load_words(w, vo, a);
        return strip_packed(a, xb, d.scale, acc);
      }
      return acc;
    }
    if constexpr (D < 4) {
      int k = 0;
      for (; k + D <= np; k += D) {
        uint2 a[D];
        strip_load_words(w, vo + 512u * k, a);
        acc = strip_packed(a, xb, d.scale, acc);
      }
      for (; k < np; ++k) {
        uint2 a[1];
        strip_load_words(w, vo + 512u * k, a);
        acc = strip_packed(a, xb, d.scale, acc);
      }
      return acc;
    }
    uint2 a[4], b[4];
    strip_load_words(w, vo, a);
    int k = 4;
    for (;;) {
      if (np - k < 4) return strip_packed_rest(w, vo, k, np, a, xb, d.scale, acc);
      strip_load_words(w, vo + 512u * k, b);
      acc = strip_packed(a, xb, d.scale, acc);
      k += 4;
      if (np - k < 4) return strip_packed_rest(w, vo, k, np, b, xb, d.scale, acc);
      strip_load_words(w, vo + 512u * k, a);
      acc = strip_packed(b, xb, d.scale, acc);
      k += 4;
    }
  }
  const size_t o = (size_t)d.off * 128;
  const X xn = x.rebase((ptrdiff_t)d.base - (1 << 15));
  if (std::is_same<typename X::value, float>::value && v32) {
    if (d.cls == kStripNear) return strip_full_sum<true, D>(S.vf + o, S.vh + o, np, lane, xn, acc);
    return strip_full_sum<false, D>(S.vf + o, S.vc + o, np, lane, x, acc);
  }
  if (d.cls == kStripNear) return strip_full_sum<true, D>(S.vv + o, S.vh + o, np, lane, xn, acc);
  return strip_full_sum<false, D>(S.vv + o, S.vc + o, np, lane, x, acc);
}

// Descriptor i (wave-uniform).
__device__ __forceinline__ StripDesc strip_desc(const StripView &S, int i) { return load_uniform(S.desc + i); }

// Bit `lane` of a wave-uniform mask.
__device__ __forceinline__ bool mask_bit(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// Adds the products of the N diagonals from q.  row >= 0; lanes without an
// entry gather their own one.
template <int N, class X>
__device__ __forceinline__ double strip_diag(const DiagSlot *q, const X &x, int row, bool v32, double acc) {
  struct Slots { DiagSlot d[N]; };
  const Slots c = load_uniform((const Slots *)q);
  typename X::value g[N];
#pragma unroll
  for (int i = 0; i < N; ++i) g[i] = x.get((uint32_t)(row + (mask_bit(c.d[i].mask) ? c.d[i].off : 0)));
#pragma unroll
  for (int i = 0; i < N; ++i)
    acc = __builtin_fma(v32 ? (double)(float)c.d[i].val : c.d[i].val, mask_bit(c.d[i].mask) ? (double)g[i] : 0.0, acc);
  return acc;
}

// Sum of the lane's entries of a strip of the diagonal class.
template <class X>
__device__ __forceinline__ double strip_diag_sum(const StripView &S, const StripDesc &d, const X &x, int row,
                                                 double own, bool v32, double acc) {
  const DiagSlot *q = S.dslot + d.off;
  const DiagSlot m = load_uniform(q);
  const int r = max(row, 0);
  acc = __builtin_fma(v32 ? (double)(float)m.val : m.val, mask_bit(m.mask) ? own : 0.0, acc);
  ++q;
  int n = d.npair;
  for (; n >= 6; n -= 6, q += 6) acc = strip_diag<6>(q, x, r, v32, acc);
  if (n >= 4) {
    acc = strip_diag<4>(q, x, r, v32, acc);
    n -= 4;
    q += 4;
  }
  if (n >= 2) {
    acc = strip_diag<2>(q, x, r, v32, acc);
    n -= 2;
    q += 2;
  }
  return n > 0 ? strip_diag<1>(q, x, r, v32, acc) : acc;
}

// Strips idx(0) .. idx(n - 1): f(strip, descriptor, row, long, sum with the
// lead, own entry of x); row -1: the lane has none; long: the row's other
// entries are in pieces.  (Loading the next strip's words and lead before the
// gathers of the current one was slower: with four word pairs a strip always
// loaded, 128^3 SpMV 17.4 -> 18.9 us, FP64 CG 28.9 -> 34.9 us an iteration.  The
// waves of a CU hide the two trips; the loads themselves are what counts.)
template <bool EARLY, int D = 4, class X, class Idx, class F>
__device__ __forceinline__ void strips_run(const StripView &S, int lane, const X &x, bool v32, int n, Idx idx, F f) {
#pragma unroll 1
  for (int k = 0; k < n; ++k) {
    const int s = idx(k);
    auto lead = [&]() { return v32 ? (double)S.lead32[64 * s + lane] : S.lead64[64 * s + lane]; };
    double ld = EARLY && S.leads ? lead() : 0.0;
    const StripDesc d = strip_desc(S, s);
    bool lng;
    const int row = strip_row(S, s, lane, lng);
    const double own = row >= 0 ? (double)x.get((uint32_t)row) : 0.0;
    double acc = 0.0;
    if ((d.flags & kStripLead) && row >= 0)
      acc = (EARLY && S.leads ? ld : lead()) * own;
    acc = d.cls == kStripDiag ? strip_diag_sum(S, d, x, row, own, v32, acc) : strip_sum<D>(S, d, x, lane, acc, v32);
    f(s, d, row, lng, acc, own);
  }
}

// Sum over the wave of a piece's products.
template <int D = 4, class X>
__device__ __forceinline__ double piece_sum(const StripView &S, int piece, int lane, const X &x, bool v32) {
  return wave_sum(strip_sum<D>(S, strip_desc(S, S.nstrips + piece), x, lane, 0.0, v32));
}

}  // namespace mf
