// The HIP runtime calls of libgeauxdock.so on the host, for tests of the
// engine's host code without a device: device memory is zeroed host memory,
// kernels are recorded and not run, and allocations and launches can be made to
// fail. Loaded with global symbols before the engine, whose calls then resolve
// here.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Launch {
  std::string kernel;
  unsigned grid[3];
  bool table;  // the complex table, its first argument, is allocated memory
};

std::map<void *, size_t> live;           // device and pinned allocations
std::vector<size_t> allocs;              // sizes asked for (failed ones too)
std::map<const void *, std::string> kernels;
std::vector<Launch> launches;
long made = 0;                           // streams and events created
long fail_alloc = -1, fail_launch = -1;  // calls until the failing one
int fill = 0;                            // what a word cleared to 0 becomes
size_t fail_above = 0;                   // every allocation above this fails (0: none)
unsigned char symbol[4 << 20];
struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} config;

hipError_t last = hipSuccess;  // of any call, until it is asked for

hipError_t allocate(void **p, size_t bytes) {
  allocs.push_back(bytes);
  *p = nullptr;
  if (fail_alloc >= 0 && fail_alloc-- == 0) return last = hipErrorOutOfMemory;
  if (fail_above > 0 && bytes > fail_above) return last = hipErrorOutOfMemory;
  *p = std::calloc(1, bytes);
  if (!*p) return last = hipErrorOutOfMemory;
  live[*p] = bytes;
  return hipSuccess;
}

hipError_t release(void *p) {
  if (!p) return hipSuccess;
  if (live.erase(p) == 0) std::abort();  // not ours, or given back twice
  std::free(p);
  return hipSuccess;
}

template <class T>
hipError_t make(T *handle) {
  made += 1;
  *handle = reinterpret_cast<T>(std::malloc(1));
  return hipSuccess;
}
template <class T>
hipError_t unmake(T handle) {
  std::free(reinterpret_cast<void *>(handle));
  return hipSuccess;
}

}  // namespace

extern "C" {

// ---- controls of the tests ----
void host_hip_fail_alloc(long n) { fail_alloc = n; }    // the n-th from now, once
void host_hip_fail_launch(long n) { fail_launch = n; }
void host_hip_fail_above(size_t bytes) { fail_above = bytes; }
void host_hip_fill(int value) { fill = value; }
long host_hip_num_allocs() { return (long)allocs.size(); }
size_t host_hip_alloc_size(long i) { return allocs[i]; }
long host_hip_num_live() { return (long)live.size(); }
long host_hip_num_made() { return made; }
long host_hip_num_launches() { return (long)launches.size(); }
const char *host_hip_kernel(long i) { return launches[i].kernel.c_str(); }
unsigned host_hip_grid(long i, int axis) { return launches[i].grid[axis]; }
int host_hip_table(long i) { return launches[i].table; }

// ---- the runtime ----
void **__hipRegisterFatBinary(const void *) {
  static void *module = nullptr;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  kernels[stub] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  config = {grid, block, lds, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  *grid = config.grid;
  *block = config.block;
  *lds = config.lds;
  *stream = config.stream;
  return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t) {
  if (!f) std::abort();
  if (fail_launch >= 0 && fail_launch-- == 0) return last = hipErrorLaunchFailure;
  // the limits of the device's grids
  if (grid.x == 0 || grid.y == 0 || grid.z == 0 || grid.y > 65535 || grid.z > 65535)
    return last = hipErrorInvalidConfiguration;
  // the table is also the first field of the MC kernels' argument block
  const std::string &name = kernels[f];
  bool table = false;
  if (name.find("gd_mc_kernel") != std::string::npos || name.find("gd_sur_feat") != std::string::npos)
    table = live.count(*static_cast<void **>(args[0])) != 0;
  launches.push_back({name, {grid.x, grid.y, grid.z}, table});
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) {
  return e == hipSuccess ? "no error" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}

hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {  // R0600 by the header's macro
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 64 * 1024;
  p->maxSharedMemoryPerMultiProcessor = 160 * 1024;
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int) {
  return f ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = symbol;
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) { return allocate(p, bytes); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(p, bytes); }
hipError_t hipFree(void *p) { return release(p); }
hipError_t hipHostFree(void *p) { return release(p); }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int value, size_t bytes, hipStream_t) {
  std::memset(dst, value, bytes);
  if (value == 0 && fill != 0)
    for (size_t i = 0; i < bytes / sizeof(int); ++i) static_cast<int *>(dst)[i] = fill;
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return unmake(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  return s && e ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventCreate(hipEvent_t *e) { return make(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return unmake(e); }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  return e ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return make(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return make(e);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return unmake(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return unmake(e); }

}  // extern "C"
