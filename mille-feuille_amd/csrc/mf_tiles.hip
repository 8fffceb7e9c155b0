// mf_tiles.hip -- device layout of the tiled matrix: upload, payload packing
// (FP32 / FP16 / INT8 copies with per-tile scales, computed on the GPU) and
// per-tile precision control.
//
// HBM layout per handle (T = tilenum, Z = nnz, ZP = payload slots: each
// tile's entries padded to a multiple of 4, so that a 4-entry chunk never
// straddles two tiles; Z <= ZP < Z + 3T):
//   tile_ptr  (tilem+1) i32    tile-row -> first tile
//   tile_col  T i32            tile column
//   tile_off  (T+1) i32        payload offset of each tile, a multiple of 4
//                              (ZP at the end)
//   tile_row  T i32            tile-row of each tile
//   tile_nz   T u8             nnz of the tile - 1
//   rc        ZP u8            (row << 4) | col of the entry inside its tile
//                              (padding repeats the tile's last byte)
//   v64/v32/v16/v8             ZP entries each (padding 0): FP64, FP32, FP16 (scaled by
//                              a power of two per tile), INT8 (scaled by a
//                              power of two per tile)
//   s16, s8   T f32            per-tile scales
//   qerr      3T f64           per-tile max |a - dequant(a)| for FP32/16/INT8
//   amax      T f64            per-tile max |a|
//   prec      T u8             current precision level of each tile
//   spmv_desc                  per-wave work (tile-rows, tiles, entries)
//                              of the stand-alone SpMV
// Entries keep the reference's order (tile by tile, row by row inside a
// tile, src/csr2block.h:239-252); the per-entry row nibble replaces the
// reference's 16 row pointers per tile on the device, so one SpMV reads
// value + 1 byte per entry and 12-16 bytes per tile.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "mf_device.h"

namespace mf {

// Payload arrays carry kPad extra zero entries: the streamed SpMV reads
// entries in aligned groups of four and may touch up to three past the end.
constexpr int kPad = 64;
constexpr int kSpmvWaveNnz = 1024;

// Host arrays of the tiles as uploaded for the packing.
struct PackSrc {
  const double *val;      // csrsize values, tile by tile
  const float *low;       // the caller's FP32 copy, or null: (float) value
  const uint8_t *col;     // column nibble of each value
  const uint8_t *ptr;     // row starts: 16 per tile, `hlast` per tile of the last tile-row
  const int *off;         // tilenum + 1 value offsets
  int tlast, hlast;       // first tile and rows of the last tile-row
};

struct PackDst {
  const int *tile_off;
  uint8_t *tile_nz, *rc, *rp16;
  double *v64;
  float *v32;
  uint16_t *v16;
  int8_t *v8;
  float *s16, *s8;
  double *qerr, *amax;
};

__device__ __forceinline__ double max16(double v) {
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) v = fmax(v, __shfl_xor(v, m));
  return v;
}

// Tile-row of every tile and the diagonal tile of every tile-row: 16 lanes
// per tile-row.
__global__ __launch_bounds__(256) void k_tile_rows(int tm, const int *__restrict__ tile_ptr,
                                                   const int *__restrict__ tile_col, int *__restrict__ tile_row,
                                                   int *__restrict__ diag) {
  const int r = blockIdx.x * 16 + (threadIdx.x >> 4);
  if (r >= tm) return;
  for (int t = tile_ptr[r] + (threadIdx.x & 15); t < tile_ptr[r + 1]; t += 16) {
    tile_row[t] = r;
    if (tile_col[t] == r) diag[r] = t;
  }
}

// Payload layout of one tile per 16 lanes, lane r packing row r: entries
// padded per tile to a multiple of 4 (zero values that repeat the tile's last
// (row,col) byte), so every 4-entry chunk of the streamed SpMV lies in one
// tile; the FP32 / FP16 / INT8 copies, their scales and errors; the 16 row
// starts (rows past the last row of a short final tile-row start at the
// tile's nnz, which is then <= 15*16) and nnz - 1.  A thread per tile took
// 0.20 ms for the 525k tiles of a 90 x 91 x 93 Laplacian, and its inputs were
// packed row by row on the host (20 ms).
__global__ __launch_bounds__(256) void k_pack_tiles(int T, PackSrc s, PackDst d) {
  const int t = blockIdx.x * 16 + (threadIdx.x >> 4), r = threadIdx.x & 15;
  if (t >= T) return;  // (alike in the 16 lanes that share a reduction)
  const int o = s.off[t], nz = s.off[t + 1] - o, po = d.tile_off[t], pz = d.tile_off[t + 1] - po;
  const int h = t >= s.tlast ? s.hlast : 16;
  const uint8_t *rp = s.ptr + (t >= s.tlast ? (size_t)s.tlast * 16 + (size_t)(t - s.tlast) * s.hlast : (size_t)t * 16);
  const int b = r < h ? rp[r] : nz, e = r < h - 1 ? rp[r + 1] : nz;
  double m = 0.0;
  for (int k = b; k < e; ++k) m = fmax(m, fabs(s.val[o + k]));
  m = max16(m);
  // FP16: power-of-two scale 2^e with e = floor(log2 max|a|), so the scaled
  // magnitudes lie in [.., 2); scaling by a power of two is exact in FP32, so
  // for in-range tiles the stored value equals (half)(float)a.
  int x = m > 0.0 ? ilogb(m) : 0;
  x = x < -100 ? -100 : (x > 100 ? 100 : x);
  const float sc16 = ldexpf(1.0f, x);
  const float inv16 = ldexpf(1.0f, -x);
  // INT8: smallest power-of-two scale with max|a|/scale <= 127 (exact
  // division; tiles of multiples of the scale, such as the -1 couplings of a
  // Laplacian, are stored exactly), round to nearest even.
  float sc8 = 1.0f;
  if (m > 0.0) {
    int x8 = ilogb(m / 127.0);
    if (ldexp(127.0, x8) < m) ++x8;
    x8 = x8 < -120 ? -120 : (x8 > 120 ? 120 : x8);
    sc8 = ldexpf(1.0f, x8);
  }
  double e32 = 0.0, e16 = 0.0, e8 = 0.0;
  for (int k = b; k < e; ++k) {
    const double v = s.val[o + k];
    const int c = s.col[o + k], i = po + k;
    d.rc[i] = (uint8_t)((r << 4) | c);
    d.v64[i] = v;
    const float f = (float)v;
    d.v32[i] = s.low ? s.low[o + k] : f;
    e32 = fmax(e32, fabs(v - (double)f));
    const _Float16 g = (_Float16)(f * inv16);
    d.v16[i] = __builtin_bit_cast(uint16_t, g);
    e16 = fmax(e16, fabs(v - (double)((float)g * sc16)));
    double q = rint(v / (double)sc8);
    q = q > 127.0 ? 127.0 : (q < -127.0 ? -127.0 : q);
    d.v8[i] = (int8_t)q;
    e8 = fmax(e8, fabs(v - q * (double)sc8));
    if (k == nz - 1)
      for (int z = nz; z < pz; ++z) {
        d.rc[po + z] = (uint8_t)((r << 4) | c);
        d.v64[po + z] = 0.0;
        d.v32[po + z] = 0.0f;
        d.v16[po + z] = 0;
        d.v8[po + z] = 0;
      }
  }
  e32 = max16(e32);
  e16 = max16(e16);
  e8 = max16(e8);
  d.rp16[(size_t)t * 16 + r] = (uint8_t)b;
  if (r == 0) {
    d.tile_nz[t] = (uint8_t)(nz - 1);
    d.s16[t] = sc16;
    d.s8[t] = sc8;
    d.amax[t] = m;
    d.qerr[t] = e32;
    d.qerr[T + t] = e16;
    d.qerr[2 * T + t] = e8;
  }
}

template <typename T>
static mf_status dalloc(T **p, size_t n) {
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    return fail(MF_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
  }
  return MF_OK;
}


mf_status upload_spmv_schedule(mf_tiled *t, int wave_nnz);

mf_status upload_tiles(mf_tiled *t, int device, const int *rowptr) {
  DeviceLayout &d = t->dev;
  MF_HIP(hipSetDevice(device));
  d.device = device;
  const int T = t->tilenum, TM = t->tilem;
  d.npad = kTile * std::max(t->tilem, t->tilen);
  if (d.npad == 0) d.npad = kTile;

  // payload offsets: each tile's entries padded to a multiple of 4
  std::vector<int> &poff = t->pay_off;
  poff.assign(T + 1, 0);
  for (int tt = 0; tt < T; ++tt) {
    const int nzt = t->csr_offset[tt + 1] - t->csr_offset[tt];
    poff[tt + 1] = poff[tt] + ((nzt + 3) & ~3);
  }
  const int ZP = poff[T];
  d.npay = ZP;
  int max_tiles = 0;
  for (int bi = 0; bi < TM; ++bi) max_tiles = std::max(max_tiles, t->tile_ptr[bi + 1] - t->tile_ptr[bi]);
  d.max_tiles_per_row = max_tiles;
  Slab slab;
  slab.add(&d.tile_ptr, TM + 1);
  slab.add(&d.tile_col, T);
  slab.add(&d.tile_off, T + 1);
  slab.add(&d.tile_row, T);
  slab.add(&d.tile_nz, T);
  slab.add(&d.rc, (size_t)ZP + kPad);
  slab.add(&d.rp16, (size_t)T * kTile + kPad);
  slab.add(&d.v64, (size_t)ZP + kPad);
  slab.add(&d.v32, (size_t)ZP + kPad);
  slab.add(&d.v16, (size_t)ZP + kPad);
  slab.add(&d.v8, (size_t)ZP + kPad);
  slab.add(&d.s16, T);
  slab.add(&d.s8, T);
  slab.add(&d.qerr, 3 * (size_t)T);
  slab.add(&d.amax, T);
  slab.add(&d.prec, T);
  slab.add(&d.prec_user, T);
  slab.add(&d.diag_tile, TM);
  MF_TRY(slab.alloc(&d.slab));
  MF_HIP(hipMemcpy(d.tile_ptr, t->tile_ptr.data(), sizeof(int) * (TM + 1), hipMemcpyHostToDevice));
  MF_HIP(hipMemcpy(d.tile_off, poff.data(), sizeof(int) * (T + 1), hipMemcpyHostToDevice));
  // the slots past the last tile that a 16-byte load may touch
  MF_HIP(hipMemset(d.rc + ZP, 0, kPad));
  MF_HIP(hipMemset(d.v64 + ZP, 0, sizeof(double) * kPad));
  MF_HIP(hipMemset(d.v32 + ZP, 0, sizeof(float) * kPad));
  MF_HIP(hipMemset(d.v16 + ZP, 0, sizeof(uint16_t) * kPad));
  MF_HIP(hipMemset(d.v8 + ZP, 0, kPad));
  if (TM > 0) MF_HIP(hipMemset(d.diag_tile, 0xff, sizeof(int) * TM));
  // per-wave work of the stand-alone SpMV, about kSpmvWaveNnz entries per
  // wave (retuned by mf_tile_set_schedule)
  MF_TRY(upload_spmv_schedule(t, kSpmvWaveNnz));
  if (T > 0) {
    MF_HIP(hipMemset(d.prec, MF_PREC_FP64, T));
    MF_HIP(hipMemset(d.prec_user, MF_PREC_FP64, T));
    MF_HIP(hipMemcpy(d.tile_col, t->tile_columnidx.data(), sizeof(int) * T, hipMemcpyHostToDevice));
    // the reference arrays, for the packing only
    double *val = nullptr;
    float *low = nullptr;
    uint8_t *col = nullptr, *ptr = nullptr;
    int *off = nullptr;
    void *tmp = nullptr;
    Slab src;
    src.add(&val, t->csrsize);
    if (t->low_given) src.add(&low, t->csrsize);
    src.add(&col, t->csrsize);
    src.add(&ptr, t->csrptrlen);
    src.add(&off, T + 1);
    MF_TRY(src.alloc(&tmp));
    auto up = [](void *q, const void *h, size_t bytes) { return hipMemcpy(q, h, bytes, hipMemcpyHostToDevice); };
    hipError_t e = up(val, t->Blockcsr_Val.data(), sizeof(double) * t->csrsize);
    if (e == hipSuccess && low) e = up(low, t->Blockcsr_Val_Low.data(), sizeof(float) * t->csrsize);
    if (e == hipSuccess) e = up(col, t->Tile_csr_Col.data(), t->csrsize);
    if (e == hipSuccess) e = up(ptr, t->Blockcsr_Ptr.data(), t->csrptrlen);
    if (e == hipSuccess) e = up(off, t->csr_offset.data(), sizeof(int) * (T + 1));
    if (e == hipSuccess) {
      k_tile_rows<<<(TM + 15) / 16, 256>>>(TM, d.tile_ptr, d.tile_col, d.tile_row, d.diag_tile);
      const PackSrc ps{val, low, col, ptr, off, t->tile_ptr[TM - 1], t->rowA - (TM - 1) * kTile};
      const PackDst pd{d.tile_off, d.tile_nz, d.rc, d.rp16, d.v64, d.v32, d.v16, d.v8, d.s16, d.s8, d.qerr, d.amax};
      k_pack_tiles<<<(T + 15) / 16, 256>>>(T, ps, pd);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    (void)hipFree(tmp);
    if (e != hipSuccess) return fail(MF_ERR_HIP, std::string("tile upload: ") + hipGetErrorString(e));
  }
  MF_TRY(build_strips(t, rowptr));
  t->strips.lean = lean_strips(t);
  t->strips.work = strip_work(t->strips);
  d.spmv_kernel = default_spmv_kernel(t);
  return MF_OK;
}

bool regular_tilerows(const mf_tiled *t) {
  const int TM = t->tilem;
  if (TM == 0) return false;
  const double mean = (double)t->tilenum / TM;
  return t->dev.max_tiles_per_row <= 4.0 * mean + 8.0;
}

int default_spmv_kernel(const mf_tiled *t) { return strips_for_product(t) ? MF_SPMV_STRIP : MF_SPMV_STREAM; }

// Stand-alone SpMV schedule of about wave_nnz payload slots per wave, heavy
// tile-rows cut into one-window pieces, uploaded in place of the previous one.
mf_status upload_spmv_schedule(mf_tiled *t, int wave_nnz) {
  DeviceLayout &d = t->dev;
  std::vector<int> hn, hbase;
  const std::vector<WaveDesc> wd = window_partition(t, wave_nnz, &hn, &hbase);
  const int nw = (int)wd.size(), nh = (int)hn.size();
  const int npieces = nh > 0 ? hbase.back() + hn.back() : 0;
  for (void *p : {(void *)d.spmv_desc, (void *)d.spmv_part, (void *)d.spmv_cnt, (void *)d.spmv_hn,
                  (void *)d.spmv_hbase})
    if (p) MF_HIP(hipFree(p));
  d.spmv_desc = nullptr;
  d.spmv_part = nullptr;
  d.spmv_cnt = nullptr;
  d.spmv_hn = d.spmv_hbase = nullptr;
  d.spmv_nwaves = 0;
  d.spmv_nheavy = 0;
  if (nw > 0) {
    MF_TRY(dalloc(&d.spmv_desc, nw));
    MF_HIP(hipMemcpy(d.spmv_desc, wd.data(), sizeof(WaveDesc) * nw, hipMemcpyHostToDevice));
  }
  MF_TRY(dalloc(&d.spmv_part, 16 * (size_t)std::max(npieces, 1)));
  MF_TRY(dalloc(&d.spmv_cnt, std::max(nh, 1)));
  MF_TRY(dalloc(&d.spmv_hn, std::max(nh, 1)));
  MF_TRY(dalloc(&d.spmv_hbase, std::max(nh, 1)));
  MF_HIP(hipMemset(d.spmv_cnt, 0, sizeof(unsigned) * std::max(nh, 1)));
  if (nh > 0) {
    MF_HIP(hipMemcpy(d.spmv_hn, hn.data(), sizeof(int) * nh, hipMemcpyHostToDevice));
    MF_HIP(hipMemcpy(d.spmv_hbase, hbase.data(), sizeof(int) * nh, hipMemcpyHostToDevice));
  }
  d.spmv_nwaves = nw;
  d.spmv_nheavy = nh;
  d.spmv_wave_nnz = wave_nnz;
  return MF_OK;
}

void free_device(mf_tiled *t) {
  DeviceLayout &d = t->dev;
  if (d.device >= 0) (void)hipSetDevice(d.device);
  void *ptrs[] = {d.slab, d.spmv_desc, d.spmv_part, d.spmv_cnt, d.spmv_hn, d.spmv_hbase, d.mlp, d.feat16,
                  t->sched.wave_tr, t->sched.wave_res, t->sched.wave_win, t->sched.win_desc, t->sched.heavy_part,
                  t->sched.heavy_cnt, t->sched.heavy_n, t->sched.heavy_base, t->sched.heavy_tr,
                  t->sched.wave_heavy, t->strip_sched.slab, t->work};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  free_strips(t);
  d = DeviceLayout();
  t->sched = Schedule();
  t->strip_sched = StripSchedule();
  t->work = nullptr;
  t->work_bytes = 0;
}

}  // namespace mf

using namespace mf;

extern "C" mf_status mf_tile_create(int rowA, int colA, const int *rowptr, const int *colidx,
                                    const double *val, const float *val_low, int device,
                                    mf_tiled **out) {
  if (!out) return fail(MF_ERR_ARG, "mf_tile_create: null output");
  *out = nullptr;
  if (device != -1) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
      return fail(MF_ERR_HIP, "mf_tile_create: no HIP device");
    if (device < 0 || device >= ndev) return fail(MF_ERR_ARG, "mf_tile_create: bad device");
  }
  mf_tiled *t = new mf_tiled();
  mf_status st = build_tiles_host(t, rowA, colA, rowptr, colidx, val, val_low);
  if (st == MF_OK && device != -1) st = upload_tiles(t, device, rowptr);
  if (device == -1) t->dev.npad = kTile * std::max(std::max(t->tilem, t->tilen), 1);
  if (st != MF_OK) {
    std::string msg = mf_last_error();
    free_device(t);
    delete t;
    set_error(msg);
    return st;
  }
  *out = t;
  return MF_OK;
}

extern "C" void mf_tile_free(mf_tiled *t) {
  if (!t) return;
  free_device(t);
  delete t;
}

extern "C" mf_status mf_tile_set_precision(mf_tiled *t, const unsigned char *levels, int uniform) {
  if (!t) return fail(MF_ERR_ARG, "mf_tile_set_precision: null handle");
  if (t->dev.device < 0) return fail(MF_ERR_ARG, "mf_tile_set_precision: host-only handle");
  MF_HIP(hipSetDevice(t->dev.device));
  const int T = t->tilenum;
  if (levels) {
    for (int i = 0; i < T; ++i)
      if (levels[i] > MF_PREC_SKIP) return fail(MF_ERR_ARG, "mf_tile_set_precision: bad level");
    MF_HIP(hipMemcpy(t->dev.prec, levels, T, hipMemcpyHostToDevice));
    MF_HIP(hipMemcpy(t->dev.prec_user, levels, T, hipMemcpyHostToDevice));
  } else {
    if (uniform < 0 || uniform > MF_PREC_SKIP) return fail(MF_ERR_ARG, "mf_tile_set_precision: bad level");
    MF_HIP(hipMemset(t->dev.prec, uniform, T));
    MF_HIP(hipMemset(t->dev.prec_user, uniform, T));
  }
  return MF_OK;
}

extern "C" mf_status mf_tile_get_precision(const mf_tiled *t, unsigned char *levels) {
  if (!t || !levels) return fail(MF_ERR_ARG, "mf_tile_get_precision: null argument");
  if (t->dev.device < 0) return fail(MF_ERR_ARG, "mf_tile_get_precision: host-only handle");
  MF_HIP(hipSetDevice(t->dev.device));
  MF_HIP(hipMemcpy(levels, t->dev.prec, t->tilenum, hipMemcpyDeviceToHost));
  return MF_OK;
}

extern "C" mf_status mf_tile_get_scales(const mf_tiled *t, float *scale16, float *scale8) {
  if (!t) return fail(MF_ERR_ARG, "mf_tile_get_scales: null handle");
  if (t->dev.device < 0) return fail(MF_ERR_ARG, "mf_tile_get_scales: host-only handle");
  MF_HIP(hipSetDevice(t->dev.device));
  if (scale16) MF_HIP(hipMemcpy(scale16, t->dev.s16, sizeof(float) * t->tilenum, hipMemcpyDeviceToHost));
  if (scale8) MF_HIP(hipMemcpy(scale8, t->dev.s8, sizeof(float) * t->tilenum, hipMemcpyDeviceToHost));
  return MF_OK;
}

extern "C" mf_status mf_tile_get_quant_error(const mf_tiled *t, double *err) {
  if (!t || !err) return fail(MF_ERR_ARG, "mf_tile_get_quant_error: null argument");
  if (t->dev.device < 0) return fail(MF_ERR_ARG, "mf_tile_get_quant_error: host-only handle");
  MF_HIP(hipSetDevice(t->dev.device));
  MF_HIP(hipMemcpy(err, t->dev.qerr, sizeof(double) * 3 * (size_t)t->tilenum, hipMemcpyDeviceToHost));
  return MF_OK;
}

extern "C" mf_status mf_tile_set_schedule(mf_tiled *t, int spmv_wave_nnz) {
  if (!t) return fail(MF_ERR_ARG, "mf_tile_set_schedule: null handle");
  if (t->dev.device < 0) return fail(MF_ERR_ARG, "mf_tile_set_schedule: host-only handle");
  if (spmv_wave_nnz == 0) return MF_OK;
  if (spmv_wave_nnz < 64 || spmv_wave_nnz > (1 << 20))
    return fail(MF_ERR_ARG, "mf_tile_set_schedule: spmv_wave_nnz out of [64, 2^20]");
  MF_HIP(hipSetDevice(t->dev.device));
  MF_HIP(hipDeviceSynchronize());
  MF_TRY(upload_spmv_schedule(t, spmv_wave_nnz));
  // the schedule is the streamed kernel's
  if (t->dev.spmv_kernel == MF_SPMV_STRIP) t->dev.spmv_kernel = MF_SPMV_STREAM;
  return MF_OK;
}
