// mf_strip_plan.cpp -- host side of the row strips (mf_strips.h): row order,
// classes, widths and long-row pieces.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <queue>
#include <vector>

#include "mf_internal.h"

namespace mf {

// Rows sorted by length inside windows of kStripWin strips (1024 rows): wide
// enough that 64 rows of about equal length come together, narrow enough that
// a strip's stores of y stay in a few cache lines.
constexpr int kStripWin = 16;
// Longest row of a sorted layout kept in its strip.
constexpr int kLongRow = 64;

void plan_strips(const mf_tiled *t, const int *rowptr, const std::vector<RowInfo> &info,
                 const std::vector<uint8_t> &ndiag, StripPlan &P) {
  const int rows = t->rowA, nstr = (16 * t->tilem + 63) / 64;
  auto len = [&](int r) { return rowptr[r + 1] - rowptr[r]; };
  // Unsorted strips where padding every row to the longest of its 64 costs
  // at most a fifth; otherwise rows are sorted inside windows.
  long long padded = 0;
#pragma omp parallel for reduction(+ : padded)
  for (int s = 0; s < nstr; ++s) {
    int m = 0;
    for (int r = 64 * s; r < std::min(rows, 64 * s + 64); ++r) m = std::max(m, len(r));
    padded += 64LL * m;
  }
  const bool sorted = (double)padded > 1.2 * t->csrsize;
  P.sorted = sorted;
  P.nstrips = nstr;
  std::vector<int> &rowmap = P.rowmap;
  std::vector<LongRow> &lrow = P.lrow;
  if (sorted) {
    P.slot.resize(rows);
    rowmap.assign((size_t)nstr * 64, -1);
    const int wrows = 64 * kStripWin;
#pragma omp parallel
    {
      std::vector<int> ord;
#pragma omp for schedule(static)
      for (int w = 0; w < (rows + wrows - 1) / wrows; ++w) {
        const int r0 = w * wrows, r1 = std::min(rows, r0 + wrows);
        ord.resize(r1 - r0);
        std::iota(ord.begin(), ord.end(), r0);
        // long rows count as empty: their entries are in pieces
        auto key = [&](int r) { return len(r) > kLongRow ? 0 : len(r); };
        std::stable_sort(ord.begin(), ord.end(), [&](int p, int q) { return key(p) > key(q); });
        for (int i = 0; i < r1 - r0; ++i) {
          P.slot[ord[i]] = r0 + i;
          rowmap[r0 + i] = ord[i] | (len(ord[i]) > kLongRow ? kLongBit : 0);
        }
      }
    }
    // long rows, those of several pieces first
    for (int many = 1; many >= 0; --many)
      for (int r = 0; r < rows; ++r)
        if (len(r) > kLongRow && (len(r) > kPieceEntries) == many) {
          if (P.long_of.empty()) {
            P.long_of.assign(rows, -1);
            P.lane_long.assign((size_t)nstr * 64, -1);
          }
          P.long_of[r] = P.lane_long[P.slot[r]] = (int)lrow.size();
          lrow.push_back(LongRow{r, P.slot[r], 0, 0});
          P.nmulti += many;
        }
    // rows past the matrix (the last tile-row's padding) keep a lane each
    for (int r = rows; r < 16 * t->tilem; ++r) rowmap[r] = r;
  }
  auto row_of = [&](int i) {  // matrix row of strip lane i, or -1
    const int r = !sorted ? i : rowmap[i] < 0 ? rows : rowmap[i] & (kLongBit - 1);
    return r < rows ? r : -1;
  };
  auto scale_of = [](int lo) { return std::ldexp(1.0f, std::max(-100, std::min(lo, 100))); };
  auto narrow = [](int lo, int hi) { return hi == -127 || (lo > -100 && hi < 100 && hi - lo <= 7); };
  auto pairs = [](int n) { return (n + 1) / 2; };
  // classes and widths
  P.desc.resize(nstr);
  P.safe.resize(nstr);
  int wide = 0;
#pragma omp parallel for reduction(max : wide)
  for (int s = 0; s < nstr; ++s) {
    int lo = 127, hi = -127, m = 0, first = -1;
    bool lead = true, packed = true, near = true, lng = false, exact = true;
    for (int i = 64 * s; i < 64 * s + 64; ++i) {
      const int r = row_of(i);
      if (r < 0) {
        lead = false;
        continue;
      }
      if (first < 0) first = r;
      lead = lead && info[r].diag;
      exact = exact && (info[r].plain & 1);
      if (sorted && len(r) > kLongRow) {
        lng = true;
        continue;
      }
      near = near && (info[r].plain & 2);
      lo = std::min<int>(lo, info[r].lo);
      hi = std::max<int>(hi, info[r].hi);
      m = std::max(m, len(r));
    }
    packed = exact && lead && narrow(lo, hi);
    // Diagonals where they are no more than the entries that rows are padded
    // to: a slot gathers x like an entry, with fewer instructions and no bytes
    // of its own (mf_strips.h has both sides).
    const int nd = ndiag[s] == 255 ? 255 : ndiag[s] & ~kDiagLead;
    const bool own_diag = ndiag[s] & kDiagLead;  // the diagonals differ: a lead
    const bool diag = !sorted && exact && (lead || !own_diag) && nd <= kMaxDiagSlots &&
                      nd <= 2 * pairs(lead ? m - 1 : m);
    if (diag) lead = own_diag;
    if (lead && m > 0) --m;
    wide = std::max(wide, m);
    StripDesc d;
    d.off = 0;
    d.npair = (uint16_t)(diag ? nd : pairs(m));
    d.cls = diag ? kStripDiag : packed ? kStripPacked : near ? kStripNear : kStripFull;
    d.flags = (uint8_t)((lng ? kStripLong : 0) | (lead ? kStripLead : 0));
    d.scale = packed && !diag ? scale_of(lo) : 1.0f;
    d.base = sorted ? s / kStripWin * kStripWin * 64 : 64 * s;
    P.desc[s] = d;
    P.safe[s] = std::max(first, 0);
  }
  if (wide > 100000) return;  // (unsorted strips of rows this long: no layout)
  for (size_t h = 0; h < lrow.size(); ++h) {
    const RowInfo &q = info[lrow[h].row];
    const bool lead = P.desc[lrow[h].lane >> 6].flags & kStripLead;
    const int n = len(lrow[h].row) - (lead ? 1 : 0);
    const bool packed = (q.plain & 1) && (lead || !q.diag) && narrow(q.lo, q.hi);
    lrow[h].first = (int)P.piece_long.size();
    lrow[h].n = (n + kPieceEntries - 1) / kPieceEntries;
    for (int k = 0; k < lrow[h].n; ++k) {
      StripDesc d;
      d.off = 0;
      d.npair = (uint16_t)pairs((std::min(n - k * kPieceEntries, kPieceEntries) + 63) / 64);
      d.cls = packed ? kStripPacked : kStripFull;
      d.flags = 0;
      d.scale = packed ? scale_of(q.lo) : 1.0f;
      d.base = lrow[h].row;
      P.desc.push_back(d);
      P.safe.push_back(lrow[h].row);
      P.piece_long.push_back((int)h);
    }
  }
  // offsets in each class's arrays
  for (StripDesc &d : P.desc) {
    uint64_t &n = d.cls == kStripPacked ? P.npacked : d.cls == kStripDiag ? P.ndiag : P.nfull;
    d.off = (uint32_t)n;
    n += d.npair + (d.cls == kStripDiag ? 1 : 0);
    P.any_full = P.any_full || (d.cls == kStripFull && d.npair > 0);
    P.any_near = P.any_near || d.cls == kStripNear;
  }
  P.ok = P.ndiag <= 0xffffffffull && P.npacked <= 0xffffffffull && P.nfull <= 0xffffffffull;
}

// Bytes that an FP64 product reads of the tiles.
static double tile_bytes(const mf_tiled *t) { return 9.0 * t->dev.npay + 13.0 * t->tilenum; }

bool lean_strips(const mf_tiled *t) {
  return t->strips.nstrips > 0 && (double)strip_bytes(t->strips) <= 1.2 * tile_bytes(t);
}

// The stand-alone FP64 product: each side takes the longer of what its bytes
// take at 5.5 TB/s and what its longest wave takes.  Streamed tiles: a wave walks
// a whole tile-row or about 1024 slots, 3.2 us for each 1024 (a tile-row of over
// 16384 is cut).  Strips: a lane walks its row, 0.12 us a pair of entries; a piece
// of a long row costs as much as 2 KB.  Fitted to 226 products of kNN graphs, bands
// and scattered rows of 6 to 700 entries, 8,000 to 500,000 rows, hot and cold:
// three that it gives to strips lose 5 to 9%, two that it keeps from them would
// gain more than 10%.  Both sides on MI355X, us, strips / streamed
// tiles, hot (cold): 128^3 Laplacian 16.0 / 30.2 (30.6 / 68.9); 160k-row kNN graph
// 5.0 / 6.2 (11.0 / 12.8), with random values 5.6 / 6.2 (14.2 / 12.7); 200k-row power law
// 25.8 / 149; bands of 48 entries a row whose longest are cut, 160k rows 29.8 / 17.3;
// of 75 random ones 23.8 / 22.6 (47.8 / 42.3); of 110, 8,000 rows 9.8 / 7.2.
bool strips_for_product(const mf_tiled *t) {
  const StripLayout &L = t->strips;
  if (!L.lean) return false;
  int slots = 0, pairs = 0;
  for (int r = 0; r < t->tilem; ++r)
    slots = std::max(slots, t->pay_off[t->tile_ptr[r + 1]] - t->pay_off[t->tile_ptr[r]]);
  for (const StripDesc &d : L.hdesc) pairs = std::max<int>(pairs, d.cls == kStripDiag ? (d.npair + 1) / 2 : d.npair);
  const double tiles = std::max(1.3 + 3.2 * std::max(1.0, std::min(slots, 16384) / 1024.0), 1.5 + tile_bytes(t) / 5.5e6);
  const double strips = std::max(1.5 + 0.12 * pairs, 1.5 + (strip_bytes(L) + 2000.0 * L.npieces) / 5.5e6);
  return 1.06 * strips <= tiles;
}

// Fitted to CG on 150 matrices (kNN graphs and bands of 6 to 700 entries a row,
// 8,000 to 1,000,000 rows) at 8 to 256 blocks, ns: an entry slot 0.24, with its
// value and column 0.29, half as much again where the rows of a strip come from
// a sorted window and its lanes gather from 64 lines; a diagonal's slot 0.12; a piece
// 56 besides its slots.  Tiles: a payload slot 0.28, a tile 0.95; under the mixed
// policies 0.13 and 2.2, which put the line where the two sides meet.
double strip_work(const StripLayout &L) {
  double ns = 56.0 * L.npieces;
  for (const StripDesc &d : L.hdesc) {
    if (d.cls == kStripDiag)
      ns += 64 * 0.12 * (d.npair + 1);
    else
      ns += 128 * d.npair * (d.cls == kStripPacked ? 0.24 : 0.29) * (L.sorted ? 1.5 : 1.0);
  }
  return 1e-3 * ns;
}

double tile_work(const mf_tiled *t, bool mixed) {
  return 1e-3 * (mixed ? 0.13 * t->dev.npay + 2.2 * t->tilenum : 0.28 * t->dev.npay + 0.95 * t->tilenum);
}

void plan_strip_schedule(const mf_tiled *t, int nwaves, StripSchedule &s) {
  const StripLayout &L = t->strips;
  s.nwaves = nwaves;
  s.wave_tr.resize(nwaves + 1);
  s.wave_piece.assign(nwaves + 1, 0);
  s.piece_order.clear();
  auto bound = [&](int w) { return (int)((long long)L.nstrips * w / nwaves); };
  for (int w = 0; w <= nwaves; ++w) s.wave_tr[w] = std::min(4 * bound(w), t->tilem);
  if (L.npieces == 0) return;
  // a strip costs its pairs and about six pairs' worth of own rows and waits
  using Load = std::pair<int, int>;
  std::priority_queue<Load, std::vector<Load>, std::greater<Load>> pq;
  for (int w = 0; w < nwaves; ++w) {
    int c = 0;
    for (int i = bound(w); i < bound(w + 1); ++i) c += 6 + L.hdesc[i].npair;
    pq.push({c, w});
  }
  std::vector<std::vector<int>> mine(nwaves);
  for (int q = 0; q < L.npieces; ++q) {
    const Load top = pq.top();
    pq.pop();
    mine[top.second].push_back(q);
    pq.push({top.first + 4 + L.hdesc[L.nstrips + q].npair, top.second});
  }
  for (int w = 0; w < nwaves; ++w) {
    s.piece_order.insert(s.piece_order.end(), mine[w].begin(), mine[w].end());
    s.wave_piece[w + 1] = (int)s.piece_order.size();
  }
}

}  // namespace mf
