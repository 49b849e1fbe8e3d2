// A HIP runtime on the host, for tests of what libtvbx.so does around its
// kernels: device memory is host memory, copies copy, kernels do nothing, and
// every launch is noted by name (a captured one as its graph is launched).
// The test can have one allocation fail.  A module's image is the text of the
// kernel names that it holds.
#include <hip/hip_runtime.h>

#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

static std::map<const void *, std::string> g_kernels;
static std::map<char *, size_t> g_mem;
static std::vector<std::string> g_log, *g_capture;
static const size_t BIG = 1u << 30;
static long g_fail = -1;  // allocations until the one that fails
static bool g_fail_on;    // and all after it

static void note(const std::string &name, unsigned gx, unsigned gy) {
  (g_capture ? *g_capture : g_log)
      .push_back(name + " " + std::to_string(gx) + "x" + std::to_string(gy));
}

extern "C" {
// the launches since the last call, one a line
const char *host_hip_log() {
  static std::string s;
  s.clear();
  for (auto &l : g_log) s += l + "\n";
  g_log.clear();
  return s.c_str();
}
// the n'th allocation from now fails (0: the next; < 0: none)
void host_hip_fail(long n) {
  g_fail = n;
  g_fail_on = false;
}
// it and all after it
void host_hip_fail_from(long n) {
  g_fail = n;
  g_fail_on = true;
}
long host_hip_left() { return g_fail; }
long host_hip_held() {
  long n = 0;
  for (auto &m : g_mem) n += (long)m.second;
  return n;
}

void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name,
                           unsigned, void *, void *, void *, void *, int *) {
  g_kernels[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static dim3 g_grid, g_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
  g_grid = g;
  g_block = b;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh,
                                     hipStream_t *st) {
  *g = g_grid;
  *b = g_block;
  *sh = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3, void **, size_t,
                           hipStream_t) {
  note(g_kernels[fn], g.x, g.y);
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy,
                                 unsigned, unsigned, unsigned, unsigned,
                                 unsigned, hipStream_t, void **, void **) {
  if (!f) return hipErrorInvalidHandle;
  note(*(std::string *)f, gx, gy);
  return hipSuccess;
}
hipError_t hipModuleLoadData(hipModule_t *m, const void *image) {
  *m = (hipModule_t) new std::string((const char *)image);
  return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t m,
                                const char *name) {
  const std::string all = " " + *(std::string *)m + " ";
  if (all.find(" " + std::string(name) + " ") == std::string::npos)
    return hipErrorNotFound;
  *f = (hipFunction_t) new std::string(name);
  return hipSuccess;
}
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(
    int *n, hipFunction_t, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipFuncGetAttribute(int *v, hipFunction_attribute, hipFunction_t) {
  *v = 1024;
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) {
  if (g_fail == 0 && g_fail_on) return hipErrorOutOfMemory;
  if (g_fail >= 0 && g_fail-- == 0) return hipErrorOutOfMemory;
  // large memory is address space only, until it is touched
  *p = n < BIG ? calloc(1, n ? n : 1)
               : mmap(nullptr, n, PROT_READ | PROT_WRITE,
                      MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  g_mem[(char *)*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  const size_t n = g_mem[(char *)p];
  g_mem.erase((char *)p);
  if (n < BIG)
    free(p);
  else
    munmap(p, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char scratch[256];
  *p = scratch;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  auto it = g_mem.upper_bound((char *)p);
  if (it == g_mem.begin()) return hipErrorInvalidValue;
  --it;
  if ((char *)p >= it->first + it->second) return hipErrorInvalidValue;
  memset(a, 0, sizeof *a);
  a->type = hipMemoryTypeDevice;
  a->devicePointer = (void *)p;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind,
                          hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp,
                            size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  for (size_t r = 0; r < h; ++r)
    memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_capture = new std::vector<std::string>;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)g_capture;
  g_capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *,
                               char *, size_t) {
  *e = (hipGraphExec_t)g;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (auto &l : *(std::vector<std::string> *)e) g_log.push_back("graph " + l);
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->totalGlobalMem = 288ull << 30;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "host_hip"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t) new int;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t) new int;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.0f;
  return hipSuccess;
}
}
