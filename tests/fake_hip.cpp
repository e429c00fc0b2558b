// A HIP runtime without a device, for tests of the library's host code: device memory is host memory, a stream is a
// list of operations that run when it is synchronised, kernels do nothing.  fake_fail(name, n) makes the n-th call of
// `name` from now on fail.  Loaded into the global scope ahead of the library, its functions are the ones called.
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

static std::map<hipStream_t, std::vector<std::function<void()>>> g_queue;
static std::map<std::string, int> g_fail;
static std::map<const void *, std::string> g_kernel;  // device function names
static std::string g_launched;  // their names, in order, one a line
static std::string g_static_name;                     // kernels with this in their name use g_static bytes of LDS
static int g_static = 0, g_max_lds = 163840;

static bool fails(const char *name) {
    auto it = g_fail.find(name);
    return it != g_fail.end() && it->second > 0 && --it->second == 0;
}
static void run(hipStream_t s) {
    auto ops = std::move(g_queue[s]);
    g_queue[s].clear();
    for (auto &f : ops) f();
}

extern "C" {
int fake_pending() {
    int n = 0;
    for (auto &q : g_queue) n += (int)q.second.size();
    return n;
}
void fake_fail(const char *name, int n) { g_fail[name] = n; }
// The kernels launched since the last call.
const char *fake_launched() {
    static std::string out;
    out.swap(g_launched);
    g_launched.clear();
    return out.c_str();
}
void fake_lds(int max_lds, const char *kernel, int bytes) {
    g_max_lds = max_lds;
    g_static_name = kernel;
    g_static = bytes;
}

void **__hipRegisterFatBinary(const void *) { return (void **)calloc(1, sizeof(void *)); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
    g_kernel[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static struct { dim3 grid, block; size_t lds; hipStream_t st; } g_config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    g_config = {grid, block, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *st) {
    *grid = g_config.grid, *block = g_config.block, *lds = g_config.lds, *st = g_config.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *k, dim3, dim3, void **, size_t, hipStream_t s) {
    g_launched += g_kernel[k] + "\n";
    g_queue[s].push_back([] {});
    return hipSuccess;
}
hipError_t hipGetLastError() { return fails("hipGetLastError") ? hipErrorLaunchFailure : hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = g_max_lds;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *k) {
    std::memset(a, 0, sizeof(*a));
    a->sharedSizeBytes = g_kernel[k].find(g_static_name) != std::string::npos ? g_static : 0;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 4;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)malloc(1);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    run(s);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)malloc(1);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    if (fails("hipMalloc")) return hipErrorOutOfMemory;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (fails("hipMemcpyAsync")) return hipErrorUnknown;
    g_queue[st].push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
}
