// A HIP runtime without a device, for tests of the library's host side on the
// CPU: "device" memory is host memory, launches are recorded and not run.
// Loaded with RTLD_GLOBAL before the library, its symbols take the place of
// the real runtime's.
//   * a freed block that was the last one gives its address to the next
//     allocation, and new memory holds 0xA5 throughout
//   * copies that the library makes to the device are kept (the last one of at
//     least fake_watch bytes), and each launch notes whether a pointer in its
//     first argument leads to those bytes, intact, in a live allocation
//   * copies to the host of as many bytes as fake_d2h was given take those
//   * streams and events have names of their own, and fake_log tells what was
//     put on which stream, a line each
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct Launch { std::string name; unsigned grid[3], block[3]; int watched; };
static std::map<const void*, std::string> names;
static std::map<char*, size_t> live;
static std::vector<Launch> launches;
static std::vector<char> watched;
static std::map<size_t, std::vector<char>> d2h;
static std::string journal;
static uintptr_t next_id = 1;
static size_t watch_min = 0;
static char *arena = nullptr, *top = nullptr;
constexpr size_t ARENA = 8ull << 30;
static dim3 cfg_grid, cfg_block;
static hipStream_t cfg_stream;

static void note(const char* what, hipStream_t s, const std::string& of) {
  journal += std::string(what) + " stream" + std::to_string((uintptr_t)s) + " " + of + "\n";
}
static std::string event_name(hipEvent_t e) { return "event" + std::to_string((uintptr_t)e); }
static char symbol[1 << 12];

extern "C" {
void fake_watch(size_t bytes) { watch_min = bytes; }
void fake_d2h(const void* p, size_t n) { d2h[n].assign((const char*)p, (const char*)p + n); }
const char* fake_log() { return journal.c_str(); }
int fake_launches() { return (int)launches.size(); }
void fake_clear() { launches.clear(); journal.clear(); }
const char* fake_name(int i) { return launches[i].name.c_str(); }
unsigned fake_grid(int i, int k) { return launches[i].grid[k]; }
int fake_intact(int i) { return launches[i].watched; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t s) {
  cfg_grid = g; cfg_block = b; cfg_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = cfg_grid; *b = cfg_block; *s = 0; *st = cfg_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t, hipStream_t st) {
  Launch l{names.count(f) ? names[f] : "?", {g.x, g.y, g.z}, {b.x, b.y, b.z}, 0};
  if (!watched.empty())
    for (int i = 0; i < 16; ++i) {
      char* p;
      memcpy(&p, (char*)args[0] + 8 * i, 8);
      for (auto& [base, size] : live)
        if (p >= base && p + watched.size() <= base + size && !memcmp(p, watched.data(), watched.size())) l.watched = 1;
    }
  launches.push_back(l);
  note("launch", st, l.name);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  if (!arena) arena = top = (char*)mmap(nullptr, ARENA, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  n = (n + 255) / 256 * 256;
  if (arena == MAP_FAILED || n > (size_t)(arena + ARENA - top)) return hipErrorOutOfMemory;
  memset(top, 0xA5, n);
  *p = top;
  live[top] = n;
  top += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = live.find((char*)p);
  if (it == live.end()) return p ? hipErrorInvalidValue : hipSuccess;
  if (it->first + it->second == top) top = it->first;
  live.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k == hipMemcpyHostToDevice && watch_min && n >= watch_min) watched.assign((const char*)s, (const char*)s + n);
  if (k == hipMemcpyDeviceToHost && d2h.count(n)) memcpy(d, d2h[n].data(), n);
  else memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = symbol; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)next_id++; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { note("wait", s, event_name(e)); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)next_id++; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)next_id++; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { note("record", s, event_name(e)); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 0; return hipSuccess; }
}
