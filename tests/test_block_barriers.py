"""Order of LDS and level-byte accesses in the solvers' shared device code,
checked on the CPU: the functions are taken from mf_device.h as they stand and
run wave by wave against memory that records every access together with the
number of block barriers its wave has passed.  Two waves that touch one word
between the same two barriers, one of them writing, are unordered.

The waves' control flow does not depend on the values, so they can run one
after another, lane 0 standing for its wave."""
import os
import re
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mille-feuille_amd", "csrc",
                      "mf_device.h")

PRELUDE = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <tuple>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_fence(...) ((void)0)
#define __hip_atomic_store(...) ((void)0)
#define __builtin_bit_cast(T, v) bit_cast_to<T>(v)
template <class T, class U> T bit_cast_to(U v) { T t; std::memcpy(&t, &v, sizeof(t)); return t; }
// words of other blocks count as arrived
#define __hip_atomic_load(...) ((unsigned long long)epoch << 32)

struct Dim { int x; };
static Dim threadIdx, blockIdx{0}, blockDim{1024}, gridDim{1};
static int interval;  // barriers that the running wave has passed
static void __syncthreads() { ++interval; }
static void lds_barrier() { ++interval; }

struct Access { int wave; bool write; };
static std::map<std::tuple<const void *, int, int>, std::vector<Access>> log_;

struct Mem { const char *name; };
struct Ref {
  const Mem *m;
  int i;
  void note(bool w) const { log_[{m, i, interval}].push_back({threadIdx.x / 64, w}); }
  operator double() const { note(false); return 1.0; }
  Ref &operator=(double) { note(true); return *this; }
};
struct Lds {
  const Mem *m;
  int off;
  Ref operator[](int i) const { return Ref{m, off + i}; }
  Lds operator+(int n) const { return Lds{m, off + n}; }
};

static double wave_sum(double v) { return v; }
static double sum_waves(Lds lds, int nw) {
  double s = 0;
  for (int i = 0; i < nw; ++i) s += lds[i];
  return s;
}
static double uniform_double(double v) { return v; }
static void drain_own_memory_ops() {}
static int sync_copies() { return 1; }
static int sync_copy() { return 0; }
struct GridSync { unsigned arrive[1][1]; };
static void wait_words(const unsigned *, int, GridSync *, unsigned) {}
static bool spin_on(unsigned &, GridSync *) { return true; }
static unsigned long long __ballot(bool v) { return v; }
constexpr int kMaxGridSum = 4, __ATOMIC_AGENT = 0;
"""

MAIN = r"""
int main() {
  Mem words{"lds"};
  int barriers = -1;
  for (int w = 0; w < 16; ++w) {
    threadIdx.x = 64 * w;
    interval = 0;
    unsigned epoch = 0;
    int slot = 0;
    GridSync gs;
    double part[64];
    unsigned long long mbox[256];
    Lds lds{&words, 0};
    double a[1] = {0}, b[2] = {0}, c[3] = {0};
    // every kind of sum after every kind of sum
    grid_sum<2>(b, part, &gs, epoch, slot, lds, nullptr);
    grid_sum_values<2>(b, mbox, &gs, epoch, lds);
    grid_sum_values<2>(b, mbox, &gs, epoch, lds);
    grid_sum<3>(c, part, &gs, epoch, slot, lds, nullptr);
    grid_sum<1>(a, part, &gs, epoch, slot, lds, nullptr);
    grid_sum_values<1>(a, mbox, &gs, epoch, lds);
    grid_sum<3>(c, part, &gs, epoch, slot, lds, nullptr);
    grid_sum_values<1>(a, mbox, &gs, epoch, lds);
    grid_sum_values<2>(b, mbox, &gs, epoch, lds);
    if (barriers >= 0 && interval != barriers) return std::printf("waves pass different numbers of barriers\n"), 2;
    barriers = interval;
  }
  int bad = 0;
  for (auto &e : log_) {
    bool write = false, two = false;
    for (const Access &x : e.second) {
      write = write || x.write;
      two = two || x.wave != e.second[0].wave;
    }
    if (write && two && bad++ < 8)
      std::printf("%s[%d]: unordered accesses after barrier %d\n", ((const Mem *)std::get<0>(e.first))->name,
                  std::get<1>(e.first), std::get<2>(e.first));
  }
  std::printf("%d accesses' words, %d unordered\n", (int)log_.size(), bad);
  return log_.size() < 100 ? 3 : bad != 0;
}
"""


def _function(text, name):
    """The definition of `name`, with its template line."""
    m = re.search(r"(template <[^\n]*>\n)?__device__ __forceinline__ [\w ]+ %s\(" % name, text)
    assert m, name
    return text[m.start():text.index("\n}\n", m.start()) + 3]


def _run(tmp_path, source):
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O0", "-w", "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_grid_sums_order_their_lds_words(tmp_path):
    text = open(HEADER).read()
    fns = "".join(_function(text, n) for n in
                  ("grid_arrive", "grid_wait", "block_sum_n", "grid_sum", "grid_sum_values"))
    fns = fns.replace("double *lds,", "Lds lds,").replace("double *lds)", "Lds lds)")
    fns, n = re.subn(r"__shared__ double (\w+)\[\w+\];", r'static Mem \1_mem{"\1"}; const Lds \1{&\1_mem, 0};', fns)
    assert n == 1
    r = _run(tmp_path, PRELUDE + fns + MAIN)
    assert r.returncode == 0, r.stdout


INFER = r"""
#include <algorithm>
#include <cstdint>
#include <cstdio>
using std::max;
using std::min;
#define __device__
#define __forceinline__ inline
constexpr int kWave = 64, MF_PREC_FP32 = 1, MF_PREC_INT8 = 3, MF_PREC_SKIP = 4;
static int open_stores;  // level bytes written since the last fence
static void __threadfence_block() { open_stores = 0; }
static unsigned long long __ballot(bool v) { return v; }
static int __shfl_xor(int v, int) { return v; }
struct Byte {
  uint8_t v = 0;
  operator int() const { return v; }
  Byte &operator=(uint8_t x) { v = x; ++open_stores; return *this; }
};
struct TileView { const int *tile_col; };
struct InferCtx { const int *w; Byte *prec_out; };
struct MlpRegs {};
typedef int half4_t;
typedef int float4_t;
static const int *classes;
static void mlp_load(const int *, int, MlpRegs &) {}
static half4_t infer_features(const InferCtx &, int t, int, int, bool) { return t; }
static float4_t mlp_eval16r(const MlpRegs &, half4_t t) { return classes[t]; }
static int mlp_argmax(float4_t c) { return c; }
"""

INFER_MAIN = r"""
template <bool CMP> int check(const int *cls, int n) {
  Byte prec[64];
  for (int t = 0; t < n; ++t) prec[t].v = 1;
  classes = cls;
  open_stores = 0;
  wave_infer_tiles<CMP>(TileView{nullptr}, InferCtx{nullptr, prec}, 0, n, 0);
  return open_stores;
}
int main() {
  int same[64], mixed[64], wide[64], bad = 0;
  for (int t = 0; t < 64; ++t) { same[t] = 2; mixed[t] = 1 + t / 16 % 3; wide[t] = 0; }
  for (const int *c : {same, mixed, wide})
    for (int n : {1, 17, 64}) {
      bad += check<true>(c, n) != 0;
      bad += check<false>(c, n) != 0;
    }
  std::printf("%d returns with unfenced level stores\n", bad);
  return bad != 0;
}
"""


def test_inferred_levels_are_fenced_before_their_reader(tmp_path):
    """The lanes that store a wave's levels are not those that read them."""
    text = open(HEADER).read()
    r = _run(tmp_path, INFER + _function(text, "wave_infer_tiles") + INFER_MAIN)
    assert r.returncode == 0, r.stdout
