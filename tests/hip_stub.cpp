// A HIP runtime without a device, for CPU tests of the library's host logic:
// loaded with RTLD_GLOBAL before the library, it takes the place of the
// runtime's functions.  Device memory is host memory, copies are done at
// once, kernels do nothing but are logged; a test sets which call fails and
// how a resident launch ends, as its device code would tell the host.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::map<const void *, std::string> g_names;       // kernel stub -> mangled name
std::map<void *, size_t> g_device, g_pinned;       // live allocations
std::string g_log;
size_t g_fail_of = 0;       // device allocations of this size fail (0: none)
int g_resident = 0;         // resident launches so far
int g_end_at = 0;           // the launch that ends so (0: none), and those after it
int g_per_cu = 1;           // workgroups a compute unit holds
unsigned g_end_as = 0;      // status written: 0 its number (taken back), else the value
unsigned g_status = 0;      // as the device holds it: written once
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;

void log(const std::string &s) { g_log += s + "\n"; }

// the status word of a resident launch: its arguments' one pinned pointer
unsigned *status_of(void *args) {
  for (int k = 0; k < 48; k++) {
    char *p;
    std::memcpy(&p, static_cast<char *>(args) + 8 * k, 8);
    for (const auto &b : g_pinned)
      if (p >= static_cast<char *>(b.first) && p < static_cast<char *>(b.first) + b.second)
        return reinterpret_cast<unsigned *>(p);
  }
  return nullptr;
}

hipError_t launch(const void *f, dim3 grid, void **args, hipStream_t stream) {
  const std::string &name = g_names[f];
  const auto has = [&](const char *s) { return name.find(s) != std::string::npos; };
  if (has("k_resident_series")) return hipSuccess;
  if (has("k_resident")) {
    g_resident++;
    log("resident " + std::to_string(grid.x));
    unsigned *const status = status_of(args[0]);
    if (g_end_at && g_resident >= g_end_at && status && !*status) *status = g_end_as ? g_end_as : unsigned(g_resident);
  } else if (has("k_step")) {  // (arguments, energy, table, s): the step is table[0] + s
    const double *table = *static_cast<const double **>(args[2]);
    log((has("k_step_il") ? "il " : "step ") + std::to_string((long long)table[0] + *static_cast<int *>(args[3])));
  } else if (has("k_interleave")) {
    log("convert");
  } else {
    log("kernel " + name);
  }
  (void)stream;
  return hipSuccess;
}
}  // namespace

extern "C" {

const char *stub_log() { return g_log.c_str(); }
void stub_clear() { g_log.clear(); }
void stub_fail_allocations_of(size_t bytes) { g_fail_of = bytes; }
// resident launch number `at` (1: the first) and later ones end with `status` (0: taken back)
void stub_end_resident(int at, unsigned status) {
  g_end_at = at;
  g_end_as = status;
}
void stub_workgroups_per_cu(int n) { g_per_cu = n; }
size_t stub_device_bytes() {
  size_t n = 0;
  for (const auto &b : g_device) n += b.second;
  return n;
}

void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, uint3 *, uint3 *, dim3 *,
                           dim3 *, int *) {
  g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_grid = grid;
  g_block = block;
  g_shared = shared;
  g_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = g_grid;
  *block = g_block;
  *shared = g_shared;
  *stream = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s) {
  return launch(f, grid, args, s);
}
hipError_t hipExtLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s, hipEvent_t,
                              hipEvent_t, int) {
  return launch(f, grid, args, s);
}

hipError_t hipMalloc(void **p, size_t n) {
  if (g_fail_of && n == g_fail_of) return hipErrorOutOfMemory;
  *p = std::calloc(n ? n : 1, 1);
  if (!*p) return hipErrorOutOfMemory;
  g_device[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (p && !g_device.erase(p)) return hipErrorInvalidValue;
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(n, 1);
  if (!*p) return hipErrorOutOfMemory;
  g_pinned[*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  g_pinned.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;  // compute units
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v) {
  log("attribute " + g_names[f] + " " + std::to_string(v));
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = g_per_cu;
  return hipSuccess;
}

// streams and events: distinct handles, waits logged
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new int);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete reinterpret_cast<int *>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  log("wait for the stream");
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  log("after another launch");
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(new int);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<int *>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
}
