// A stand-in for the HIP runtime's host calls, for tests of the library's host
// code without a GPU: memory is host memory, streams and events are nothing,
// and a launch runs no kernel.  Loaded with global symbols before the
// library, whose calls then come here.  What the tests rely on is kept as
// documented: a launch with more than 64 KB of dynamic LDS needs the limit
// raised for its kernel on the current device, and a failed launch is what
// hipGetLastError reports.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <utility>
#include <vector>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
int g_device = 0, g_last = 0;
bool g_refuse_launches = false;
std::set<std::pair<int, const void *>> g_raised;
std::map<std::pair<int, const void *>, void *> g_symbols;
Dim3 g_grid, g_block;
size_t g_lds;
void *g_stream;
int g_nargs = 0;
std::vector<uint64_t> g_log;
void *handle(void **p) { return *p = calloc(1, 8); }
}  // namespace

extern "C" {
void host_set_device(int d) { g_device = d; }
void host_refuse_launches(int on) { g_refuse_launches = on != 0; }
// the first nargs arguments (8 bytes each) of every launch from now on
void host_record(int nargs) {
  g_nargs = nargs;
  g_log.clear();
}
int host_recorded(uint64_t *out, int most) {
  int n = 0;
  for (; n < most && n < (int)g_log.size(); ++n) out[n] = g_log[n];
  return (int)g_log.size();
}

int hipGetDevice(int *d) {
  *d = g_device;
  return 0;
}
int hipMalloc(void **p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? 0 : 2; }
int hipFree(void *p) {
  free(p);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  memcpy(d, s, n);
  return 0;
}
int hipMemset(void *p, int v, size_t n) {
  memset(p, v, n);
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t n, void *) {
  memset(p, v, n);
  return 0;
}
int hipGetSymbolAddress(void **p, const void *sym) {
  void *&m = g_symbols[{g_device, sym}];
  if (!m) m = calloc(1, 1 << 16);
  *p = m;
  return 0;
}
int hipFuncSetAttribute(const void *f, int, int) {
  g_raised.insert({g_device, f});
  return 0;
}
int hipLaunchKernel(const void *f, Dim3, Dim3, void **args, size_t lds, void *) {
  if (g_refuse_launches || (lds > 65536 && !g_raised.count({g_device, f}))) return g_last = 1;
  for (int i = 0; i < g_nargs; ++i) g_log.push_back(*static_cast<uint64_t *>(args[i]));
  return 0;
}
unsigned __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void *st) {
  g_grid = g;
  g_block = b;
  g_lds = lds;
  g_stream = st;
  return 0;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *lds, void **st) {
  *g = g_grid;
  *b = g_block;
  *lds = g_lds;
  *st = g_stream;
  return 0;
}
int hipGetLastError() {
  const int e = g_last;
  g_last = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e ? "refused" : "no error"; }
int hipStreamCreateWithFlags(void **s, unsigned) { return handle(s) ? 0 : 2; }
int hipStreamDestroy(void *s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipStreamIsCapturing(void *, int *status) { return *status = 0; }
int hipEventCreate(void **e) { return handle(e) ? 0 : 2; }
int hipEventCreateWithFlags(void **e, unsigned) { return handle(e) ? 0 : 2; }
int hipEventDestroy(void *e) {
  free(e);
  return 0;
}
int hipEventRecord(void *, void *) { return 0; }
}
