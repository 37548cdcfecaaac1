// A stand-in for the HIP runtime, for tests of the host side without a GPU: kernels are
// noted by name and not run, graphs hold names, device memory is host memory that is never
// touched unless it is copied.  Loaded with RTLD_GLOBAL before libmgpu.so it takes the
// place of the runtime's symbols.  fake_* below are the tests' handles.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::map<const void *, std::string> names;   // host stub -> mangled kernel name
std::map<void *, size_t> device, pinned;     // live allocations
std::vector<std::string> ran;                // kernels that ran, in order
std::vector<std::string> *capture = nullptr; // where a capture puts them
std::vector<const void *> pending;           // pageable host memory of copies in flight
std::string fail_at;                         // call or kernel to fail, once
hipError_t last = hipSuccess;
size_t to_host = 0;                          // bytes copied from the device
struct Cfg { dim3 g, b; size_t sh; hipStream_t st; };
std::vector<Cfg> cfgs;

bool fails(const char *what) {
  if (fail_at.empty() || !strstr(what, fail_at.c_str())) return false;
  fail_at.clear();
  last = hipErrorUnknown;
  return true;
}
hipError_t map_memory(void **p, size_t n, std::map<void *, size_t> &to) {
  *p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) return hipErrorOutOfMemory;
  to[*p] = n ? n : 1;
  return hipSuccess;
}
hipError_t unmap(void *p, std::map<void *, size_t> &from) {
  auto it = from.find(p);
  if (it == from.end()) return hipErrorInvalidValue;
  munmap(p, it->second);
  from.erase(it);
  return hipSuccess;
}
bool inside(const void *p, const std::map<void *, size_t> &m) {
  auto it = m.upper_bound((void *)p);
  return it != m.begin() && (--it, (const char *)p < (const char *)it->first + it->second);
}
template <class T>
hipError_t handle(T *h) {
  *h = (T)new char[8];
  return hipSuccess;
}
}  // namespace

extern "C" {
// ---- the tests' handles
void fake_reset() { ran.clear(); to_host = 0; }
void fake_fail(const char *what) { fail_at = what; }
int fake_ran(const char *kernel) {
  int n = 0;
  for (auto &s : ran) n += s.find(kernel) != std::string::npos;
  return n;
}
long fake_to_host() { return (long)to_host; }
int fake_pending() { return (int)pending.size(); }

// ---- registration and launches
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  cfgs.push_back({g, b, sh, st});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
  *g = cfgs.back().g, *b = cfgs.back().b, *sh = cfgs.back().sh, *st = cfgs.back().st;
  cfgs.pop_back();
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
  if (fails(names[f].c_str())) return last;
  (capture ? *capture : ran).push_back(names[f]);
  return hipSuccess;
}
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "an error asked for by the test"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int v) { return v <= 163840 ? hipSuccess : hipErrorInvalidValue; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return hipSuccess; }

// ---- device
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize() { pending.clear(); return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->totalGlobalMem = 288ull << 30;
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 163840;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = 288ull << 30; return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void **p, size_t n) { return map_memory(p, n, device); }
hipError_t hipFree(void *p) { return p ? unmap(p, device) : hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return map_memory(p, n, pinned); }
hipError_t hipHostFree(void *p) { return p ? unmap(p, pinned) : hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static void *scratch = nullptr;
  if (!scratch && map_memory(&scratch, (size_t)16 << 20, device) != hipSuccess) return hipErrorOutOfMemory;
  *p = scratch;
  return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (fails("hipMemcpyAsync")) return last;
  const void *host = k == hipMemcpyHostToDevice ? s : d;
  if (!inside(host, pinned)) pending.push_back(host);
  if (k == hipMemcpyDeviceToHost) to_host += n;
  memcpy(d, s, n);
  return hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { delete[] (char *)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { pending.clear(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete[] (char *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { pending.clear(); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capture = new std::vector<std::string>();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)capture;
  capture = nullptr;
  return fails("hipStreamEndCapture") ? last : hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (std::vector<std::string> *)g; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  if (fails("hipGraphInstantiate")) return last;
  *x = (hipGraphExec_t) new std::vector<std::string>(*(std::vector<std::string> *)g);
  return hipSuccess;
}
hipError_t hipGraphExecUpdate(hipGraphExec_t x, hipGraph_t g, hipGraphNode_t *, hipGraphExecUpdateResult *r) {
  *(std::vector<std::string> *)x = *(std::vector<std::string> *)g;
  *r = hipGraphExecUpdateSuccess;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete (std::vector<std::string> *)x; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
  if (fails("hipGraphLaunch")) return last;
  for (auto &s : *(std::vector<std::string> *)x) ran.push_back(s);
  return hipSuccess;
}
}
