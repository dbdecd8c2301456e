// A HIP runtime that runs nothing, for tests of the library's host side on a
// machine without a GPU: loaded with RTLD_GLOBAL before libhypno_hip.so, its
// functions stand in for the runtime's.  It writes down every kernel launch
// (name and grid) and device allocation, can be told to run out of memory and
// to report streams as under graph capture, where it refuses allocations and
// synchronisations as the runtime does.  Device addresses are host memory.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
constexpr int kOutOfMemory = 2, kCaptureUnsupported = 900;
std::map<const void*, std::string> g_names;
std::map<void*, size_t> g_live;
std::string g_log;
size_t g_used = 0, g_limit = ~(size_t)0;
int g_capturing = 0, g_last = 0;
Dim3 g_grid, g_block;
size_t g_lds;
void* g_stream;
int fail(int e) { return g_last = e; }
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  g_names[fn] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  g_grid = grid;
  g_block = block;
  g_lds = lds;
  g_stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = g_grid;
  *block = g_block;
  *lds = g_lds;
  *stream = g_stream;
  return 0;
}
int hipLaunchKernel(const void* fn, Dim3 grid, Dim3 block, void**, size_t lds, void*) {
  char line[64];
  snprintf(line, sizeof line, " %u %u %u\n", grid.x, grid.y, grid.z);
  // (what the hardware has: 160 KB of LDS and 1024 threads a work-group)
  if (lds > 160 * 1024 || block.x * block.y * block.z > 1024) return fail(1);
  g_log += "launch " + g_names[fn] + line;
  return 0;
}
int hipMalloc(void** p, size_t n) {
  if (g_capturing) return fail(kCaptureUnsupported);
  if (n > g_limit || g_used > g_limit - n) return fail(kOutOfMemory);
  *p = aligned_alloc(256, 256);  // (nothing is read or written through it)
  g_live[*p] = n;
  g_used += n;
  g_log += "malloc " + std::to_string(n) + "\n";
  return 0;
}
int hipFree(void* p) {
  auto it = g_live.find(p);
  if (it == g_live.end()) return fail(1);
  g_log += "free " + std::to_string(it->second) + "\n";
  g_used -= it->second;
  g_live.erase(it);
  free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return (*p = malloc(n)) ? 0 : fail(kOutOfMemory); }
int hipHostFree(void* p) { return free(p), 0; }
int hipHostGetDevicePointer(void** d, void* p, unsigned) { return *d = p, 0; }
int hipMemcpy(void*, const void*, size_t, int) { return 0; }
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = malloc(1), 0; }
int hipStreamDestroy(void* s) { return free(s), 0; }
int hipStreamSynchronize(void*) { return g_capturing ? fail(kCaptureUnsupported) : 0; }
int hipDeviceSynchronize() { return g_capturing ? fail(kCaptureUnsupported) : 0; }
int hipStreamIsCapturing(void*, int* status) { return *status = g_capturing, 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = malloc(1), 0; }
int hipEventDestroy(void* e) { return free(e), 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, 0; }  // (256 CUs)
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  return *n = 1, 0;
}
int hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), 0; }
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetLastError() {
  const int e = g_last;
  g_last = 0;
  return e;
}

const char* fake_log() {
  static std::string out;
  out.swap(g_log);
  g_log.clear();
  return out.c_str();
}
void fake_set_capturing(int on) { g_capturing = on; }
void fake_set_room(size_t bytes) { g_limit = bytes == ~(size_t)0 ? bytes : g_used + bytes; }
int fake_last_error() { return g_last; }
}
