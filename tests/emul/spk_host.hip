// A stand-in for the HIP runtime, linked with libspk_hip's own sources as
// host code (tests/emul/libspk_host.so): the library's host side (which
// kernels a call launches, what it allocates, what it does when an
// allocation fails) runs on the CPU.  Kernels do nothing: device memory is
// zeroed host memory, a launch is a line of the log, a captured graph is the
// lines its replay writes.  tests/test_host_cpu.py drives it through the C ABI
// and the spk_host_* calls below.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

extern "C" {
char __hip_fatbin[64];   // what the sources' registration would point at
}

namespace {

struct Block {
  size_t bytes;
};
std::map<void *, Block> g_device, g_host;
size_t g_device_bytes, g_device_limit, g_free_reported, g_total = (size_t)288 << 30;
long g_device_calls, g_host_calls;
int g_fail_host, g_fail_info;
hipError_t g_last = hipSuccess;
std::vector<std::string> g_log;
bool g_capturing;
std::vector<std::string> *g_capture;
long g_execs, g_captures;
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;

hipError_t fail(hipError_t e) { return g_last = e; }

// (the sources register their kernels before this file's own objects exist)
std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}

void note(std::string s) { (g_capturing ? *g_capture : g_log).push_back(std::move(s)); }

struct Graph {
  std::vector<std::string> lines;
};

}  // namespace

extern "C" {

// ------------------------------------------------------------- test's calls
void spk_host_reset(void) {
  g_device_limit = 0;
  g_free_reported = 0;
  g_fail_host = g_fail_info = 0;
  g_last = hipSuccess;
  g_log.clear();
}
// device allocations fail beyond this many live bytes (0: no limit)
void spk_host_limit(size_t bytes) { g_device_limit = bytes; }
void spk_host_free_memory(size_t bytes) { g_free_reported = bytes; }   // what hipMemGetInfo reports (0: the rest)
void spk_host_fail_pinned(int n) { g_fail_host = n; }                  // the next n pinned allocations fail
void spk_host_fail_info(int n) { g_fail_info = n; }                    // the next n hipMemGetInfo calls fail
size_t spk_host_device_bytes(void) { return g_device_bytes; }
long spk_host_device_calls(void) { return g_device_calls; }
long spk_host_pinned_calls(void) { return g_host_calls; }
long spk_host_execs(void) { return g_execs; }                          // graphs that are held
long spk_host_captures(void) { return g_captures; }
// the launches since the last call, one a line: name, workgroups, threads
const char *spk_host_log(void) {
  static std::string s;
  s.clear();
  for (auto &l : g_log) s += l + "\n";
  g_log.clear();
  return s.c_str();
}

// ------------------------------------------------------------------ runtime
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  int status = 0;
  char *p = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  std::string s = p && !status ? p : name;
  std::free(p);
  for (const char *cut : {"(anonymous namespace)::", "void ", "spk::"})
    for (size_t at; (at = s.find(cut)) != std::string::npos;) s.erase(at, std::strlen(cut));
  const size_t at = s.rfind(">(") != std::string::npos ? s.rfind(">(") + 1 : s.find('(');
  names()[host] = s.substr(0, at);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_grid = grid, g_block = block, g_shared = shared, g_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = g_grid, *block = g_block, *shared = g_shared, *stream = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
  note(names()[f] + " " + std::to_string(grid.x) + " " + std::to_string(block.x));
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) {
  g_device_calls++;
  if (g_capturing) return fail(hipErrorStreamCaptureUnsupported);
  if (g_device_limit && g_device_bytes + n > g_device_limit) return fail(hipErrorOutOfMemory);
  *p = std::calloc(n ? n : 1, 1);
  if (!*p) return fail(hipErrorOutOfMemory);
  g_device[*p] = Block{n};
  g_device_bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = g_device.find(p);
  if (it == g_device.end()) return p ? fail(hipErrorInvalidValue) : hipSuccess;
  g_device_bytes -= it->second.bytes;
  g_device.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  g_host_calls++;
  if (g_fail_host > 0) {
    g_fail_host--;
    return fail(hipErrorOutOfMemory);
  }
  *p = std::calloc(n ? n : 1, 1);
  g_host[*p] = Block{n};
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  auto it = g_host.find(p);
  if (it == g_host.end()) return p ? fail(hipErrorInvalidValue) : hipSuccess;
  g_host.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
  if (g_fail_info > 0) {
    g_fail_info--;
    return fail(hipErrorInvalidValue);
  }
  *total = g_total;
  *free_bytes = g_free_reported ? g_free_reported : g_total - g_device_bytes;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
  std::memset(p, v, n);
  return hipSuccess;
}

const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) {   // kept until it is read, whatever succeeds meanwhile
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}

hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeSharedMemPerBlockOptin ? 160 << 10 : 64 << 10;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char rows[1 << 20];
  *p = rows;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipStreamCreate(hipStream_t *s) {
  *s = reinterpret_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  return g_capturing ? fail(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_capturing = true;
  g_captures++;
  g_capture = new std::vector<std::string>();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  g_capturing = false;
  *g = reinterpret_cast<hipGraph_t>(new Graph{std::move(*g_capture)});
  delete g_capture;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(g)));
  g_execs++;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<Graph *>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete reinterpret_cast<Graph *>(e);
  g_execs--;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (auto &l : reinterpret_cast<Graph *>(e)->lines) g_log.push_back(l);
  return hipSuccess;
}

}  // extern "C"
