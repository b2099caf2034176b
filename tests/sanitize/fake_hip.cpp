// A HIP runtime without a GPU, preloaded in place of the real one: device
// memory is host memory, kernels do nothing (the build flags are written, with
// a largest row that the test chooses), one allocation can be made to fail, and
// every launch of a kernel named below is checked for pointers that are null
// or already freed.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

std::mutex mu;
std::map<char *, size_t> live;                // allocation -> size
std::map<const void *, std::string> kernels;  // host function -> name
int fail_in = 0, rows = 40;
long bad = 0, launches = 0, mallocs = 0;
bool scanned = false;

// kernel name -> arguments that have to point into live memory
const std::vector<std::pair<const char *, std::vector<int>>> kPointers = {
    {"k_b_load", {1, 2, 3, 5, 6, 7, 8}},
    {"k_b_scatter", {3, 4}},
    {"k_b_build", {1, 2, 5, 11, 12}},
    {"k_b_ljI", {2, 6, 7, 9}},
    {"k_b_lj_vjp", {2, 5, 6, 8, 9, 10}},
    {"k_b_eam_rho", {1, 5, 9, 10, 11}},
    {"k_b_eam_force", {1, 5, 9, 10, 11}},
    {"k_b_eam_adj_a", {1, 4, 8, 9, 10, 11, 13, 14}},
    {"k_b_eam_adj_b", {1, 4, 9}},
    {"k_b_colsum_chunks", {0, 7}},
    {"k_b_colsumE", {0, 3}},
    {"k_wrap_bin", {1, 2, 3, 4, 5, 6}},
    {"k_scan_bins", {1, 2}},
    {"k_bin_scatter", {1, 3, 4, 5}},
    {"k_build_group", {1, 4, 5, 6}},
    {"k_ljI", {7, 10, 11, 13, 14}},
    {"k_eam_rho", {7, 10, 11, 12}},
    {"k_eam_force", {7, 10, 11, 12, 16}},
};

bool is_live(const void *p) {
  auto it = live.upper_bound((char *)p);
  return it != live.begin() && (char *)p < std::prev(it)->first + std::prev(it)->second;
}

hipError_t launched(const void *fn, void **args) {
  std::lock_guard<std::mutex> lock(mu);
  launches++;
  const std::string &name = kernels[fn];
  if (name.find("k_build_flags") != std::string::npos) {
    int *host = *(int **)args[1];
    host[0] = rows;
    host[15] = *(int *)args[2];
    return hipSuccess;
  }
  if (name.find("rocprim") != std::string::npos) scanned = true;
  if (name.find("k_b_load") != std::string::npos) scanned = false;
  if (name.find("k_b_scatter") != std::string::npos && name.find("k_b_scatter_g") == std::string::npos && !scanned) {
    std::fprintf(stderr, "%s without a scan before it\n", name.c_str());
    bad++;
  }
  for (auto &k : kPointers)
    if (name.find(k.first) != std::string::npos && name.find("k_b_scatter_g") == std::string::npos)
      for (int a : k.second)
        if (!is_live(*(void **)args[a])) {
          std::fprintf(stderr, "%s: argument %d is %p\n", name.c_str(), a, *(void **)args[a]);
          bad++;
        }
  return hipSuccess;
}

hipError_t take(void **p, size_t n) {
  std::lock_guard<std::mutex> lock(mu);
  mallocs++;
  *p = nullptr;
  if (fail_in > 0 && --fail_in == 0) return hipErrorOutOfMemory;
  *p = std::calloc(n ? n : 1, 1);
  live[(char *)*p] = n ? n : 1;
  return hipSuccess;
}

hipError_t give(void *p) {
  std::lock_guard<std::mutex> lock(mu);
  if (!p) return hipSuccess;
  if (!live.erase((char *)p)) {
    std::fprintf(stderr, "free of %p\n", p);
    bad++;
    return hipErrorInvalidValue;
  }
  std::free(p);
  return hipSuccess;
}

}  // namespace

extern "C" {
// ---- for the test
void fake_fail_in(int n) { fail_in = n; }
void fake_rows(int n) { rows = n; }
long fake_bad() { return bad; }
long fake_launches() { return launches; }
long fake_mallocs() { return mallocs; }

// ---- the runtime
void **__hipRegisterFatBinary(const void *) { return (void **)std::calloc(1, sizeof(void *)); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  kernels[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
static thread_local Call call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
  call = {g, b, s, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
  *g = call.grid, *b = call.block, *s = call.lds, *st = call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **args, size_t, hipStream_t) { return launched(fn, args); }
hipError_t hipExtLaunchKernel(const void *fn, dim3, dim3, void **args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
  return launched(fn, args);
}
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t *, size_t *, hipDeviceptr_t) { return hipErrorInvalidValue; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char symbol[64];
  *p = symbol;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { return std::memset(a, 0, sizeof(*a)), hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 64, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->sharedMemPerBlock = 65536;
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
}
