// The HIP runtime functions that libmillefeuille_hip.so calls, on host memory,
// for CPU tests of the library's host code: allocations come from a budget,
// kernels are logged and not run but for the fill (device memory starts at
// zero), asynchronous copies happen at the next synchronisation, and event times follow a cost per
// kernel name.  Loaded with RTLD_GLOBAL before the library, so the library's calls
// resolve here.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <cxxabi.h>
#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 { uint32_t x, y, z; };
struct Copy { void *dst; const void *src; std::vector<char> then; int kind; };
constexpr int kFill = -1;  // (of dst, then.size() bytes, with the word in src)
std::map<const void *, std::string> names;
std::map<void *, size_t> live;
std::vector<Copy> queue;
std::string log_;
std::vector<std::pair<std::string, float>> costs;
size_t in_use, budget = SIZE_MAX;
int stale, last_error;
double clock_us;
Dim3 cfg_grid, cfg_block;
alignas(256) char symbol[12 << 20];

void drain() {
  for (Copy &c : queue) {
    if (c.kind == kFill) {
      for (size_t i = 0; i < c.then.size(); i += 4) std::memcpy((char *)c.dst + i, &c.src, 4);
      continue;
    }
    if (c.kind == 1 && std::memcmp(c.src, c.then.data(), c.then.size())) ++stale;
    std::memcpy(c.dst, c.kind == 1 ? c.then.data() : c.src, c.then.size());
  }
  queue.clear();
}

int launch(const void *f, Dim3 grid, void **args) {
  const std::string &n = names[f];
  log_ += "launch " + n + " " + std::to_string(grid.x) + "\n";
  float us = 1.0f;
  for (auto &c : costs)
    if (n.find(c.first) != std::string::npos) us = c.second;
  clock_us += us;
  if (n == "mf::k_fill_u32")
    queue.push_back({*(void **)args[0], (const void *)(uintptr_t)*(uint32_t *)args[2],
                     std::vector<char>(4 * *(size_t *)args[1]), kFill});
  return 0;
}
}  // namespace

extern "C" {
// for the tests
const char *fake_log() { return log_.c_str(); }
void fake_clear() { log_.clear(); }
void fake_budget(size_t bytes) { budget = bytes; }
size_t fake_in_use() { return in_use; }
int fake_stale_copies() { return stale; }
void fake_cost(const char *kernel, float us) { costs.push_back({kernel, us}); }

void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  int st = 0;
  char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  std::string s = d && !st ? d : name;
  std::free(d);
  if (s.rfind("void ", 0) == 0) s = s.substr(5);
  const std::string anon = "(anonymous namespace)::";
  for (size_t i; (i = s.find(anon)) != std::string::npos;) s.erase(i, anon.size());
  // the arguments' list, after the template's
  int depth = 0;
  for (size_t i = 0; i < s.size(); ++i) {
    if (s[i] == '<') ++depth;
    if (s[i] == '>') --depth;
    if (s[i] == '(' && depth == 0) { s = s.substr(0, i); break; }
  }
  for (size_t i; (i = s.find(' ')) != std::string::npos;) s.erase(i, 1);
  names[f] = s;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t, void *) { cfg_grid = g; cfg_block = b; return 0; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *m, void **s) {
  *g = cfg_grid;
  *b = cfg_block;
  *m = 0;
  *s = nullptr;
  return 0;
}
int hipLaunchKernel(const void *f, Dim3 g, Dim3, void **a, size_t, void *) { return launch(f, g, a); }
int hipLaunchCooperativeKernel(const void *f, Dim3 g, Dim3, void **a, unsigned, void *) { return launch(f, g, a); }

int hipMalloc(void **p, size_t n) {
  log_ += "malloc " + std::to_string(n) + "\n";
  if (n > budget - in_use) { *p = nullptr; return last_error = 2; }
  if (!(*p = std::calloc(1, n + 256))) return last_error = 2;
  live[*p] = n;
  in_use += n;
  return 0;
}
int hipFree(void *p) {
  if (!p) return 0;
  drain();
  auto it = live.find(p);
  if (it == live.end()) return last_error = 1;
  in_use -= it->second;
  live.erase(it);
  std::free(p);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) { drain(); std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) {
  queue.push_back({d, s, std::vector<char>((const char *)s, (const char *)s + n), kind});
  return 0;
}
int hipMemset(void *d, int v, size_t n) { drain(); std::memset(d, v, n); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *) { drain(); std::memset(d, v, n); return 0; }
int hipDeviceSynchronize() { drain(); return 0; }
int hipStreamSynchronize(void *) { drain(); return 0; }
int hipStreamCreate(void **s) { *s = (void *)8; return 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamBeginCapture(void *, int) { return 0; }
int hipStreamEndCapture(void *, void **g) { *g = (void *)8; return 0; }
int hipGraphInstantiate(void **e, void *, void *, char *, size_t) { *e = (void *)8; return 0; }
int hipGraphLaunch(void *, void *) { return 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
int hipEventCreate(void **e) { *e = new double(0); return 0; }
int hipEventDestroy(void *e) { delete (double *)e; return 0; }
int hipEventRecord(void *e, void *) { *(double *)e = clock_us; return 0; }
int hipEventSynchronize(void *) { drain(); return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { *ms = (float)(*(double *)b - *(double *)a) * 1e-3f; return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return 0; }
int hipGetSymbolAddress(void **p, const void *) { *p = symbol; return 0; }
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
}
