// The HIP runtime calls of the library as host functions that record what they are asked for and launch
// nothing, so that its host code (launch shapes, error paths, ordering of streams) runs without a GPU.
//
// Loaded with RTLD_GLOBAL before the library, whose undefined HIP symbols then resolve to it.  Device memory is
// host memory that starts as 0xAA bytes; memory of more than 64 MiB is neither filled, set nor copied (only the
// calls are recorded).  A launch is refused as HIP refuses it: an empty grid, or 2^32 work-items in a dimension.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
constexpr size_t kReal = 64u << 20;
std::string g_log;
std::map<const void*, std::string> g_names;           // host stub -> kernel
std::map<std::string, std::pair<int, int>> g_fail;     // call -> (calls until it fails, error)
hipError_t g_last = hipSuccess;
hipStream_t g_capturing = (hipStream_t)-1;  // the stream that records a graph
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
struct {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} g_cfg;

void note(const std::string& s) { g_log += s + "\n"; }
std::string hex(const void* p) {
  char b[32];
  std::snprintf(b, sizeof b, "%p", p);
  return b;
}
hipError_t set(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
bool fails(const char* fn, hipError_t* e) {
  auto it = g_fail.find(fn);
  if (it == g_fail.end() || --it->second.first > 0) return false;
  *e = (hipError_t)it->second.second;
  g_fail.erase(it);
  note(std::string("failed ") + fn);
  g_last = *e;
  return true;
}
}  // namespace

#define IEQ_MAY_FAIL(fn) \
  hipError_t err;        \
  if (fails(fn, &err)) return err

extern "C" {

const char* host_hip_log() { return g_log.c_str(); }
void host_hip_clear() { g_log.clear(); }
void host_hip_fail(const char* fn, int nth, int code) { g_fail[fn] = {nth, code}; }  // the nth call from now on
void host_hip_capture(void* s) { g_capturing = (hipStream_t)s; }
int host_hip_last() { return (int)g_last; }

void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  g_cfg = {g, b, sh, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
  *g = g_cfg.grid;
  *b = g_cfg.block;
  *sh = g_cfg.shared;
  *s = g_cfg.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s) {
  IEQ_MAY_FAIL("hipLaunchKernel");
  char t[160];
  std::snprintf(t, sizeof t, " %u %u %u %u %u %u %p", g.x, g.y, g.z, b.x, b.y, b.z, (void*)s);
  const bool ok = g.x && g.y && g.z && (unsigned long long)g.x * b.x < (1ull << 32) && (unsigned long long)g.y * b.y < (1ull << 32) &&
                  (unsigned long long)g.z * b.z < (1ull << 32);
  note((ok ? "launch " : "refused ") + g_names[f] + t);
  return ok ? hipSuccess : set(hipErrorInvalidConfiguration);
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "recorded error"; }

hipError_t hipMalloc(void** p, size_t n) {
  IEQ_MAY_FAIL("hipMalloc");
  *p = std::malloc(n ? n : 1);
  if (n <= kReal) std::memset(*p, 0xAA, n);
  note("malloc " + hex(*p) + " " + std::to_string(n) + (g_mode == hipStreamCaptureModeRelaxed ? " relaxed" : ""));
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  note("free " + hex(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  IEQ_MAY_FAIL("hipHostMalloc");
  *p = std::malloc(n);
  std::memset(*p, 0xAA, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = 288ull << 30;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  IEQ_MAY_FAIL("hipMemsetAsync");
  note("memset " + hex(p) + " " + std::to_string(n) + " " + hex(s));
  if (n <= kReal) std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { return hipMemsetAsync(p, v, n, nullptr); }
hipError_t hipMemcpyAsync(void* d, const void* a, size_t n, hipMemcpyKind, hipStream_t s) {
  IEQ_MAY_FAIL("hipMemcpyAsync");
  note("memcpy " + hex(d) + " " + hex(a) + " " + std::to_string(n) + " " + hex(s));
  if (n <= kReal) std::memcpy(d, a, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* a, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, a, n, k, nullptr); }

hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* a, size_t ap, size_t w, size_t h, hipMemcpyKind, hipStream_t s) {
  IEQ_MAY_FAIL("hipMemcpyAsync");
  note("memcpy " + hex(d) + " " + hex(a) + " " + std::to_string(w * h) + " " + hex(s));
  if (dp * h <= kReal && ap * h <= kReal)
    for (size_t k = 0; k < h; ++k) std::memcpy((char*)d + k * dp, (const char*)a + k * ap, w);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)std::malloc(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  IEQ_MAY_FAIL("hipStreamSynchronize");
  note("synchronize " + hex(s));
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  IEQ_MAY_FAIL("hipStreamWaitEvent");
  note("wait " + hex(s) + " " + hex(e));
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  IEQ_MAY_FAIL("hipStreamIsCapturing");
  *st = g_capturing == s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  const hipStreamCaptureMode old = g_mode;
  g_mode = *m;
  *m = old;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  IEQ_MAY_FAIL("hipEventCreate");
  *e = (hipEvent_t)std::malloc(8);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  note("record " + hex(e) + " " + hex(s));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = nullptr;
  return hipErrorInvalidValue;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return hipSuccess;
}

}  // extern "C"
