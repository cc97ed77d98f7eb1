// A stand-in for the HIP runtime, for tests of the engine's host code on the CPU:
// loaded before libvegas_hip.so with its symbols global, it takes the engine's
// calls.  Device memory is host memory, kernels are not run, and every call that
// bears on order is one line of a log.  A test can make the nth call of a
// function fail, leave an error for hipGetLastError, and bound the device memory.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include <hip/hip_runtime_api.h>

namespace {
std::map<const void*, std::string> g_kernels;
std::map<const void*, size_t> g_sizes;
std::map<std::string, int> g_fail;  // calls until the failing one
std::string g_log;
hipError_t g_last = hipSuccess;
int g_last_in = 0;  // launches until g_last is set
size_t g_used = 0, g_limit = ~(size_t)0;
uintptr_t g_handle = 1;
int g_device = 0;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_config;

std::mutex g_mu;
void note(const std::string& s) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_log += s + "\n";
}
std::string num(const void* p) { return std::to_string((uintptr_t)p); }
// Whether this call of `fn` is the one to fail.
bool fails(const char* fn) {
    auto it = g_fail.find(fn);
    return it != g_fail.end() && it->second > 0 && --it->second == 0;
}
hipError_t bad(hipError_t e) { return g_last = e; }
template <class H>
hipError_t handle(H* out) {
    *out = (H)g_handle++;
    return hipSuccess;
}
}  // namespace

extern "C" {
// For the tests.
void fake_fail(const char* fn, int nth) { g_fail[fn] = nth; }
void fake_error_at_launch(int nth) { g_last_in = nth; }  // 0: none
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_used() { return g_used; }
const char* fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }

// Kernels.
void** __hipRegisterFatBinary(const void*) {
    static void* p = nullptr;
    return &p;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
    g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    g_config = {grid, block, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    *grid = g_config.grid;
    *block = g_config.block;
    *lds = g_config.lds;
    *st = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t st) {
    note("launch " + g_kernels[f] + " stream " + num(st) + " grid " + std::to_string(grid.x) +
         " block " + std::to_string(block.x));
    if (g_last_in > 0 && --g_last_in == 0) g_last = hipErrorLaunchFailure;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 4;
    return hipSuccess;
}

// Devices and errors.
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = g_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "made to fail"; }

// Memory.
hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (fails("hipMalloc") || g_used + n > g_limit) return bad(hipErrorOutOfMemory);
    *p = std::calloc(1, n);
    g_sizes[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = g_sizes.find(p);
    if (it != g_sizes.end()) {
        g_used -= it->second;
        g_sizes.erase(it);
        std::free(p);
    }
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    note("hostmalloc " + std::to_string(n));
    *p = nullptr;
    if (fails("hipHostMalloc")) return bad(hipErrorOutOfMemory);
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) {
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t st) {
    note("copy stream " + num(st) + " bytes " + std::to_string(n));
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* mem = std::calloc(1, 64u << 20);
    *p = mem;
    return hipSuccess;
}

// Streams, events, graphs.
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    if (fails("hipStreamCreateWithFlags")) return bad(hipErrorOutOfMemory);
    const hipError_t e = handle(s);
    note("stream " + num(*s));
    return e;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    note("sync stream " + num(s));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (fails("hipStreamWaitEvent")) return bad(hipErrorUnknown);
    note("wait stream " + num(s) + " event " + num(e));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (fails("hipEventCreateWithFlags")) return bad(hipErrorOutOfMemory);
    return handle(e);
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (fails("hipEventRecord")) return bad(hipErrorUnknown);
    note("record event " + num(e) + " stream " + num(s));
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return handle(e);
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t st) {
    note("graph stream " + num(st));
    return hipSuccess;
}
}
