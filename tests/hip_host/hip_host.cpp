// The part of the HIP runtime that libmeshstage.so calls, over host memory of a stated size and with launches that only leave
// their kernel's name and grid behind: what the library allocates, gives back and launches can then be checked without a GPU.
// Loaded (RTLD_GLOBAL) before libmeshstage.so, whose references bind to it.  Test infrastructure, never shipped.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex mu;
size_t total_bytes = (size_t)1 << 32, used_bytes = 0;
long long others = 0, take_after_info = 0;              // held by other processes; taken by them behind the next hipMemGetInfo
std::map<void *, size_t> blocks;
std::map<const void *, std::string> kernels;
std::string launches, scratch;
thread_local hipError_t last_error = hipSuccess;
hipError_t result(hipError_t e) {
    if (e != hipSuccess) last_error = e;
    return e;
}
size_t free_bytes() {
    const long long f = (long long)total_bytes - (long long)used_bytes - others;
    return f > 0 ? (size_t)f : 0;
}
int dummy;
}  // namespace

extern "C" {

// ---- what a test asks and sets
void host_memory(size_t total) { std::lock_guard<std::mutex> l(mu); total_bytes = total; }
void host_others(long long bytes) { std::lock_guard<std::mutex> l(mu); others = bytes; }
void host_take_after_info(long long bytes) { std::lock_guard<std::mutex> l(mu); take_after_info = bytes; }
size_t host_used() { std::lock_guard<std::mutex> l(mu); return used_bytes; }
// the launches since the last call, a line each: mangled name, grid x, y, z, threads
const char *host_launches() {
    std::lock_guard<std::mutex> l(mu);
    scratch.swap(launches);
    launches.clear();
    return scratch.c_str();
}

// ---- the runtime
void **__hipRegisterFatBinary(const void *) { static void *h[1]; return h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, uint3 *, uint3 *, dim3 *, dim3 *, int *) { kernels[host] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::mutex> l(mu);
    *p = nullptr;
    if (bytes > free_bytes()) return result(hipErrorOutOfMemory);
    *p = aligned_alloc(256, (bytes + 255) / 256 * 256 + 256);        // (what the runtime promises)
    memset(*p, 0, bytes);
    blocks[*p] = bytes;
    used_bytes += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> l(mu);
    if (!p) return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end()) return result(hipErrorInvalidValue);
    used_bytes -= it->second;
    blocks.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    std::lock_guard<std::mutex> l(mu);
    *f = free_bytes();
    *t = total_bytes;
    others += take_after_info;
    take_after_info = 0;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { *p = calloc(1, bytes ? bytes : 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
    for (size_t i = 0; i < h; ++i) memcpy(static_cast<char *>(d) + i * dp, static_cast<const char *>(s) + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { static char room[16 << 20]; *p = room; return hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : result(hipErrorInvalidDevice); }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) { *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(static_cast<void *>(p), 0, sizeof *p);
    strcpy(p->name, "host memory");
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = total_bytes;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t) {
    std::lock_guard<std::mutex> l(mu);
    char dims[96];
    snprintf(dims, sizeof dims, " %u %u %u %u\n", g.x, g.y, g.z, b.x * b.y * b.z);
    launches += kernels[f] + dims;
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t smem, hipStream_t s, hipEvent_t, hipEvent_t, int) {
    return hipLaunchKernel(f, g, b, args, smem, s);
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(&dummy); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = reinterpret_cast<hipGraph_t>(&dummy); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = reinterpret_cast<hipGraphExec_t>(&dummy); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(&dummy); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }

}  // extern "C"
