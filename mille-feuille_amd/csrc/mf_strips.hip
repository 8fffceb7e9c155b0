// mf_strips.hip -- builds the row strips of a handle on the GPU from its
// uploaded tiles (a wave per row; 0.8 ms for 762k rows and 5.3M entries), and
// the stand-alone product over them.
#include <algorithm>
#include <string>
#include <vector>

#include "mf_strips.h"

namespace mf {

namespace {

// Lane's entries of row r in tile t: [b, e) of the tile's payload.
__device__ __forceinline__ void tile_row_range(const TileView &A, int t, int r, int &b, int &e) {
  b = A.rp16[(size_t)t * 16 + r];
  e = r < 15 ? A.rp16[(size_t)t * 16 + r + 1] : A.tile_nz[t] + 1;
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = min(v, __shfl_xor(v, m));
  return v;
}

// One wave per row, lanes over the tiles of its tile-row.
__global__ __launch_bounds__(256) void k_row_info(TileView A, int rows, RowInfo *__restrict__ info) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int R = row >> 4, r = row & 15;
  int lo = 127, hi = -127, diag = 0, plain = 1, far = 0;
  for (int t = A.tile_ptr[R] + lane; t < A.tile_ptr[R + 1]; t += kWave) {
    int b, e;
    tile_row_range(A, t, r, b, e);
    const int c0 = A.tile_col[t] << 4;
    for (int k = A.tile_off[t] + b; k < A.tile_off[t] + e; ++k) {
      const int c = c0 + (A.rc[k] & 15);
      const double v = A.v64[k];
      far = far || c - row > kNearCols || row - c > kNearCols;
      plain = plain && A.v32[k] == (float)v && fabs(v) < 1e30 && c - row < (1 << 22) && row - c < (1 << 22);
      if (c == row && !diag) {
        diag = 1;
        continue;
      }
      if (v == 0.0) continue;
      const uint64_t u = __builtin_bit_cast(uint64_t, v);
      const int ex = (int)((u >> 52) & 2047) - 1023;
      const uint64_t m = (u & 0xfffffffffffffull) | 0x10000000000000ull;
      lo = min(lo, ex < -100 ? -127 : ex - 52 + (int)__builtin_ctzll(m));
      hi = max(hi, ex > 100 ? 127 : ex + 1);
    }
  }
  lo = max(wave_min(lo), -127);
  hi = -wave_min(-hi);
  plain = (__ballot(!plain) == 0 ? 1 : 0) | (__ballot(far) == 0 ? 2 : 0);
  diag = __ballot(diag) != 0;
  if (lane == 0) info[row] = RowInfo{(int8_t)lo, (int8_t)hi, (uint8_t)diag, (uint8_t)plain};
}

// One wave per strip of 64 consecutive rows, a row per lane: merges the rows'
// entries (in tile order) by column - row, smallest first, so each step takes
// one entry of every row that has that offset next.  Entries are taken once
// each whatever their order; where one step's values differ, the strip has no
// diagonal form.  FILL: the slots (and leads) of the strips that the plan gave
// this class; else the number of off-diagonal slots (255: none), plus
// kDiagLead if the diagonal entries differ.
template <bool FILL>
__global__ __launch_bounds__(256) void k_diag_slots(TileView A, int rows, int nstrips, uint8_t *__restrict__ count,
                                                    const StripDesc *__restrict__ desc,
                                                    DiagSlot *__restrict__ out, double *__restrict__ lead64,
                                                    float *__restrict__ lead32) {
  const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= nstrips) return;
  if (FILL) {
    if (desc[s].cls != kStripDiag) return;
    out += desc[s].off;
  }
  const int row = 64 * s + lane, r = row & 15;
  int t = 0, tend = 0, k = 0, e = 0;
  if (row < rows) {
    t = A.tile_ptr[row >> 4];
    tend = A.tile_ptr[(row >> 4) + 1];
  }
  if (t < tend) {
    int b;
    tile_row_range(A, t, r, b, e);
    k = A.tile_off[t] + b;
    e += A.tile_off[t];
  }
  bool diag = false, live = true;
  double dv = 0.0, v = 0.0;
  int off = 0;
  auto next = [&]() {  // the lane's next off-diagonal entry
    for (;;) {
      while (k >= e && t + 1 < tend) {
        int b;
        ++t;
        tile_row_range(A, t, r, b, e);
        k = A.tile_off[t] + b;
        e += A.tile_off[t];
      }
      if (k >= e) {
        live = false;
        return;
      }
      off = (A.tile_col[t] << 4) + (A.rc[k] & 15) - row;
      v = A.v64[k];
      ++k;
      if (off != 0 || diag) return;
      diag = true;
      dv = v;
    }
  };
  // all lanes: whether the lanes of `in` hold one value, and that value
  auto common = [&](unsigned long long in, double x, double &c) {
    c = in ? __shfl(x, (int)__builtin_ctzll(in)) : 0.0;
    const bool same = __builtin_bit_cast(unsigned long long, x) == __builtin_bit_cast(unsigned long long, c);
    return (__ballot(!same) & in) == 0;
  };
  next();
  int n = 0;
  double c;
  for (unsigned long long act; (act = __ballot(live)) != 0;) {
    const int m = wave_min(live ? off : 0x7fffffff);
    const bool mine = live && off == m;
    const unsigned long long in = __ballot(mine);
    if (n == kMaxDiagSlots || !common(in, v, c)) {
      n = 255;
      break;
    }
    ++n;
    if (FILL && lane == 0) out[n] = DiagSlot{in, c, m, 0};
    if (mine) next();
  }
  const unsigned long long in = __ballot(diag);
  const bool same = common(in, dv, c);
  if (FILL) {
    const bool lead = desc[s].flags & kStripLead;
    if (lane == 0) out[0] = lead ? DiagSlot{0, 0.0, 0, 0} : DiagSlot{in, c, 0, 0};
    if (lead) {
      lead64[row] = dv;
      lead32[row] = (float)dv;  // (the payload of the rows of this class)
    }
  } else if (lane == 0) {
    count[s] = (uint8_t)(n == 255 ? n : n | (same ? 0 : kDiagLead));
  }
}

struct FillArgs {
  TileView A;
  const StripDesc *desc;
  const int *slot;      // strip lane of each row (64 s + lane), null: the row itself
  const int *long_of;   // long row of each row or -1, null: none
  const LongRow *lrow;
  uint32_t *words;
  double *vv;
  float *vf;
  int *vc;
  uint16_t *vh;
  double *lead64;
  float *lead32;
  int rows, nstrips;
};

// Entry p of strip lane `lane` (or of a piece's entry order) at descriptor d.
__device__ __forceinline__ void put_entry(const FillArgs &a, const StripDesc &d, int lane, int p, int col, double v,
                                          float f) {
  const size_t i = (size_t)d.off * 128 + (size_t)(p >> 1) * 128 + 2 * lane + (p & 1);
  if (d.cls == kStripPacked) {
    const int q = (int)(v / (double)d.scale);  // exact: v = q * scale
    a.words[i] = (uint32_t)(col - d.base + (1 << 23)) << 8 | (uint32_t)(q + 128);
  } else {
    a.vv[i] = v;
    a.vf[i] = f;
    if (d.cls == kStripNear)
      a.vh[i] = (uint16_t)(col - d.base + (1 << 15));
    else
      a.vc[i] = col;
  }
}

// One wave per row: its entries in tile order to the strip lane (or pieces)
// of the row; padding was filled before.
__global__ __launch_bounds__(256) void k_fill_strips(FillArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= a.rows) return;
  const TileView &A = a.A;
  const int R = row >> 4, r = row & 15;
  const int slot = a.slot ? a.slot[row] : row;
  const int h = a.long_of ? a.long_of[row] : -1;
  const StripDesc sd = a.desc[slot >> 6];
  if (sd.cls == kStripDiag) return;
  const bool lead = sd.flags & kStripLead;  // the diagonal goes to the lead
  const int piece0 = h >= 0 ? a.lrow[h].first : 0;
  int pos = 0;  // off-diagonal (or all) entries before this batch of tiles
  for (int t0 = A.tile_ptr[R]; t0 < A.tile_ptr[R + 1]; t0 += kWave) {
    const int t = t0 + lane;
    int b = 0, e = 0, dk = -1, c0 = 0, o = 0;
    if (t < A.tile_ptr[R + 1]) {
      tile_row_range(A, t, r, b, e);
      c0 = A.tile_col[t] << 4;
      o = A.tile_off[t];
      if (lead && A.tile_col[t] == R)
        for (int k = e - 1; k >= b; --k)
          if ((A.rc[o + k] & 15) == r) dk = k;
    }
    const int n = e - b - (dk >= 0 ? 1 : 0);
    int inc = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(inc, d);
      if (lane >= d) inc += u;
    }
    int p = pos + inc - n;
    pos += __builtin_amdgcn_readlane(inc, 63);
    for (int k = b; k < e; ++k) {
      const double v = A.v64[o + k];
      const float f = A.v32[o + k];
      if (k == dk) {
        a.lead64[slot] = v;
        a.lead32[slot] = f;
        continue;
      }
      const int col = c0 + (A.rc[o + k] & 15);
      if (h < 0) {
        put_entry(a, sd, slot & 63, p, col, v, f);
      } else {
        // piece entries go round the lanes: entry q of a piece to lane q % 64
        const int pc = p / kPieceEntries, q = p % kPieceEntries;
        put_entry(a, a.desc[a.nstrips + piece0 + pc], q & 63, q >> 6, col, v, f);
      }
      ++p;
    }
  }
}

// Padding of a strip's packed entries: the word of "no entry" with a column
// that exists.  One block per descriptor.
__global__ __launch_bounds__(256) void k_pad_words(const StripDesc *__restrict__ desc, const int *__restrict__ safe,
                                                   uint32_t *__restrict__ words) {
  const StripDesc d = desc[blockIdx.x];
  if (d.cls != kStripPacked) return;
  const uint32_t w = (uint32_t)(safe[blockIdx.x] - d.base + (1 << 23)) << 8;
  for (int i = threadIdx.x; i < 128 * d.npair; i += 256) words[(size_t)d.off * 128 + i] = w;
}

// y of a long row from the sum of its pieces.
__device__ __forceinline__ void store_long(const StripView &S, const LongRow &lr, double sum,
                                           const double *__restrict__ x, double *__restrict__ y) {
  if (S.desc[lr.lane >> 6].flags & kStripLead) sum = __builtin_fma(S.lead64[lr.lane], x[lr.row], sum);
  y[lr.row] = sum;
}

// y = A x over strips.  Blocks [0, pblocks): the long rows, a block for each
// row of several pieces (its waves take the pieces in turn, and their sums
// are added in piece order through LDS), then a wave for each row of one;
// these are the longer jobs and start first, dealt round the XCDs.  The other
// blocks: a strip per wave, each XCD a contiguous eighth of them.
template <bool PIECES>
__global__ __launch_bounds__(256, 8) void k_spmv_strip(StripView S, int pblocks, const double *__restrict__ x,
                                                       double *__restrict__ y) {
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int b = blockIdx.x;
  if (PIECES && b < pblocks) {
    if (b < S.nmulti) {
      __shared__ double part[4];
      const LongRow lr = S.lrow[b];
      double sum = 0.0;
      for (int k0 = 0; k0 < lr.n; k0 += 4) {
        double v = 0.0;
        if (k0 + wv < lr.n)
          v = piece_sum(S, lr.first + k0 + wv, lane, MemVec<double>{x}, false);
        __syncthreads();
        if (lane == 0) part[wv] = v;
        __syncthreads();
        sum += ((part[0] + part[1]) + part[2]) + part[3];
      }
      if (threadIdx.x == 0) store_long(S, lr, sum, x, y);
    } else {
      const int h = S.nmulti + (b - S.nmulti) * 4 + wv;
      if (h >= S.nlong) return;
      const LongRow lr = S.lrow[h];
      const double v = piece_sum(S, lr.first, lane, MemVec<double>{x}, false);
      if (lane == 0) store_long(S, lr, v, x, y);
    }
    return;
  }
  if (PIECES) b -= pblocks;
  const int per_xcd = (gridDim.x - (PIECES ? pblocks : 0)) >> 3;  // both counts are multiples of 8
  const int s = ((b & 7) * per_xcd + (b >> 3)) * 4 + wv;
  if (s >= S.nstrips) return;
  strips_run<true>(S, lane, MemVec<double>{x}, false, 1, [&](int) { return s; },
             [&](int, const StripDesc &, int row, bool lng, double acc, double) {
               if (row >= 0 && !lng) y[row] = acc;
             });
}

template <typename T>
mf_status upload(T *d, const std::vector<T> &h) {
  if (!h.empty()) MF_HIP(hipMemcpy(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
  return MF_OK;
}

}  // namespace

mf_status launch_spmv_strip(const mf_tiled *t, const double *d_x, double *d_y, hipStream_t s) {
  const StripView S = strip_view_of(t);
  const int sblocks = ((S.nstrips + 3) / 4 + 7) / 8 * 8;
  const int pblocks = (S.nmulti + (S.nlong - S.nmulti + 3) / 4 + 7) / 8 * 8;
  if (S.nlong > 0)
    k_spmv_strip<true><<<pblocks + sblocks, 256, 0, s>>>(S, pblocks, d_x, d_y);
  else
    k_spmv_strip<false><<<sblocks, 256, 0, s>>>(S, 0, d_x, d_y);
  MF_HIP(hipGetLastError());
  return MF_OK;
}

void free_strips(mf_tiled *t) {
  StripLayout &s = t->strips;
  if (s.slab) (void)hipFree(s.slab);
  s = StripLayout();
}

int64_t strip_bytes(const StripLayout &L) {
  int64_t b = (int64_t)(sizeof(StripDesc) * L.hdesc.size()) + (L.sorted ? 256 * (int64_t)L.nstrips : 0);
  for (const StripDesc &d : L.hdesc) {
    if (d.flags & kStripLead) b += 8 * 64;
    if (d.cls == kStripDiag)
      b += (int64_t)sizeof(DiagSlot) * (d.npair + 1);
    else
      b += 128 * (int64_t)d.npair * (d.cls == kStripPacked ? 4 : d.cls == kStripNear ? 10 : 12);
  }
  return b;
}

// (no_memory: an allocation failed for want of memory, with MF_OK returned)
static mf_status make_strips(mf_tiled *t, const int *rowptr, bool &no_memory) {
  auto alloc = [&](Slab &s, void **base) {
    const hipError_t e = s.try_alloc(base);
    if (e == hipSuccess) return MF_OK;
    *base = nullptr;
    if (e != hipErrorOutOfMemory) return fail(MF_ERR_HIP, std::string("build_strips: ") + hipGetErrorString(e));
    (void)hipGetLastError();
    no_memory = true;
    return MF_OK;
  };
  StripLayout &L = t->strips;
  const int rows = t->rowA;
  if (rows == 0 || t->tilenum == 0) return MF_OK;
  const TileView A = view_of(t);
  const int nstrips = (16 * t->tilem + 63) / 64;
  std::vector<RowInfo> info(rows);
  std::vector<uint8_t> ndiag(nstrips);
  {
    RowInfo *d = nullptr;
    uint8_t *nd = nullptr;
    Slab both;
    void *mem = nullptr;
    both.add(&d, rows);
    both.add(&nd, nstrips);
    MF_TRY(alloc(both, &mem));
    if (no_memory) return MF_OK;
    k_row_info<<<(rows + 3) / 4, 256>>>(A, rows, d);
    k_diag_slots<false><<<(nstrips + 3) / 4, 256>>>(A, rows, nstrips, nd, nullptr, nullptr, nullptr, nullptr);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpy(info.data(), d, sizeof(RowInfo) * rows, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(ndiag.data(), nd, nstrips, hipMemcpyDeviceToHost);
    (void)hipFree(mem);
    if (e != hipSuccess) return fail(MF_ERR_HIP, std::string("build_strips: ") + hipGetErrorString(e));
  }
  StripPlan P;
  plan_strips(t, rowptr, info, ndiag, P);
  if (!P.ok) return MF_OK;
  const int nstr = P.nstrips;
  const uint64_t np = P.npacked, nf = P.nfull;
  L.sorted = P.sorted;
  L.npieces = (int)P.piece_long.size();
  L.nlong = (int)P.lrow.size();
  L.nmulti = P.nmulti;
  L.hdesc = P.desc;
  int leads = 0;
  for (int s = 0; s < nstr; ++s) leads += (P.desc[s].flags & kStripLead) != 0;
  L.leads = 2 * leads >= nstr;
  int *d_safe = nullptr, *d_slot = nullptr, *d_long = nullptr;
  // (few calls: on a handle of 512 rows the strips' allocations, fills and
  // launches took 100 of 393 us)
  Slab slab, tmp;
  slab.add(&L.desc, P.desc.size());
  slab.add(&d_safe, P.safe.size());
  slab.add(&L.words, 128 * np);
  if (P.any_full) slab.add(&L.vc, 128 * nf);
  if (P.ndiag) slab.add(&L.dslot, P.ndiag);
  if (P.sorted) slab.add(&L.rowmap, P.rowmap.size());
  if (L.nlong > 0) {
    slab.add(&L.lane_long, P.lane_long.size());
    slab.add(&L.lrow, P.lrow.size());
    slab.add(&L.piece_long, P.piece_long.size());
  }
  // zero where nothing is stored: from lead64 to the end
  slab.add(&L.lead64, 64 * (size_t)nstr);
  slab.add(&L.lead32, 64 * (size_t)nstr);
  slab.add(&L.vv, 128 * nf);
  slab.add(&L.vf, 128 * nf);
  if (P.any_near) slab.add(&L.vh, 128 * nf);
  if (P.sorted) tmp.add(&d_slot, P.slot.size());
  if (L.nlong > 0) tmp.add(&d_long, P.long_of.size());
  void *scratch = nullptr;  // temporaries of the fill
  MF_TRY(alloc(slab, &L.slab));
  if (!no_memory && P.sorted) MF_TRY(alloc(tmp, &scratch));
  if (no_memory) return MF_OK;
  bool fill = false;
  for (const StripDesc &d : P.desc) fill = fill || d.cls != kStripDiag;
  if (fill) MF_HIP(hipMemset(L.lead64, 0, (size_t)((char *)L.slab + slab.bytes() - (char *)L.lead64)));
  if (L.vc && nf > 0) MF_HIP(hipMemset(L.vc, 0xff, sizeof(int) * 128 * nf));
  mf_status st = upload(L.desc, P.desc);
  if (st == MF_OK && np > 0) st = upload(d_safe, P.safe);
  if (st == MF_OK && P.sorted) st = upload(L.rowmap, P.rowmap);
  if (st == MF_OK && P.sorted) st = upload(d_slot, P.slot);
  if (st == MF_OK && L.nlong > 0) {
    st = upload(L.lane_long, P.lane_long);
    if (st == MF_OK) st = upload(L.lrow, P.lrow);
    if (st == MF_OK) st = upload(L.piece_long, P.piece_long);
    if (st == MF_OK) st = upload(d_long, P.long_of);
  }
  if (st == MF_OK) {
    if (np > 0) k_pad_words<<<(unsigned)P.desc.size(), 256>>>(L.desc, d_safe, L.words);
    FillArgs a{A, L.desc, d_slot, d_long, L.lrow, L.words, L.vv, L.vf, L.vc, L.vh,
               L.lead64, L.lead32, rows, nstr};
    if (fill) k_fill_strips<<<(rows + 3) / 4, 256>>>(a);
    if (P.ndiag) k_diag_slots<true><<<(nstr + 3) / 4, 256>>>(A, rows, nstr, nullptr, L.desc, L.dslot, L.lead64, L.lead32);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) st = fail(MF_ERR_HIP, std::string("build_strips: ") + hipGetErrorString(e));
  }
  if (scratch) (void)hipFree(scratch);
  if (st == MF_OK) L.nstrips = nstr;
  return st;
}

// Without memory for them a handle has no strips and runs on its tiles.
mf_status build_strips(mf_tiled *t, const int *rowptr) {
  bool no_memory = false;
  const mf_status st = make_strips(t, rowptr, no_memory);
  if (no_memory) free_strips(t);
  return st;
}

}  // namespace mf

using namespace mf;

extern "C" mf_status mf_tile_strip_info(const mf_tiled *t, int *strips, int *pieces, int *sorted,
                                        int64_t *packed_slots, int64_t *full_slots,
                                        int64_t *diag_slots, int64_t *bytes, int *lean) {
  if (!t) return fail(MF_ERR_ARG, "mf_tile_strip_info: null handle");
  const StripLayout &L = t->strips;
  int64_t n[3] = {0, 0, 0};
  if (L.nstrips > 0)
    for (const StripDesc &d : L.hdesc) {
      if (d.cls == kStripDiag)
        n[2] += 64 * ((int64_t)d.npair + 1);
      else
        n[d.cls == kStripPacked ? 0 : 1] += 128 * (int64_t)d.npair;
    }
  if (strips) *strips = L.nstrips;
  if (pieces) *pieces = L.npieces;
  if (sorted) *sorted = L.sorted;
  if (packed_slots) *packed_slots = n[0];
  if (full_slots) *full_slots = n[1];
  if (diag_slots) *diag_slots = n[2];
  if (bytes) *bytes = L.nstrips > 0 ? strip_bytes(L) : 0;
  if (lean) *lean = L.lean;
  return MF_OK;
}
