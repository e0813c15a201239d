// The HIP calls of libcudatracer.so on host memory, for tests of its host path
// on machines without a GPU: what it allocates, copies, waits for and launches
// is recorded, single calls can be made to fail, and kernels do nothing.  Loaded
// with RTLD_GLOBAL before the library, so that its calls bind to these.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

namespace {

std::recursive_mutex mu;
std::map<char*, size_t> device, pinned;  // allocations
size_t used, peak, capacity = (size_t)1 << 40;
std::map<std::string, int> calls, failing;
std::vector<std::pair<char*, size_t>> copies;  // destinations
hipError_t last = hipSuccess;
struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} config;
int handles;

// Counts the call; an error stays the last one until it is asked for.
hipError_t done(const char* name, hipError_t e = hipSuccess) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    ++calls[name];
    if (failing[name] > 0) {
        --failing[name];
        e = hipErrorInvalidValue;
    }
    if (e != hipSuccess) last = e;
    return e;
}
template <class T>
hipError_t handle(const char* name, T* h) {
    const hipError_t e = done(name);
    *h = e == hipSuccess ? reinterpret_cast<T>((size_t)16 * (size_t)++handles) : nullptr;
    return e;
}
bool inside(const std::map<char*, size_t>& m, const void* p) {
    char* c = static_cast<char*>(const_cast<void*>(p));
    auto it = m.upper_bound(c);
    return it != m.begin() && c < std::prev(it)->first + std::prev(it)->second;
}
hipError_t copy(const char* name, void* dst, const void* src, size_t n) {
    const hipError_t e = done(name);
    if (e != hipSuccess) return e;
    std::lock_guard<std::recursive_mutex> lk(mu);
    copies.emplace_back(static_cast<char*>(dst), n);
    std::memcpy(dst, src, n);
    return e;
}

}  // namespace

extern "C" {

// ---- for the tests
int standin_calls(const char* name) { return calls[name]; }
void standin_fail(const char* name, int times) { failing[name] = times; }
void standin_capacity(size_t bytes) { capacity = bytes; }
size_t standin_used() { return used; }
size_t standin_peak(int reset) {
    if (reset) peak = used;
    return peak;
}
// Bytes that copies have written to [p, p + n) since the last call.
size_t standin_copied(const char* p, size_t n) {
    size_t sum = 0;
    for (const auto& c : copies)
        if (c.first >= p && c.first < p + n) sum += c.second;
    copies.clear();
    return sum;
}

// ---- memory
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = nullptr;
    const hipError_t e = done("hipMalloc", used + n > capacity ? hipErrorOutOfMemory : hipSuccess);
    if (e != hipSuccess) return e;
    *p = std::calloc(n ? n : 1, 1);
    device[static_cast<char*>(*p)] = n;
    used += n;
    peak = used > peak ? used : peak;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    auto it = device.find(static_cast<char*>(p));
    if (it != device.end()) {
        used -= it->second;
        device.erase(it);
        std::free(p);
    }
    return done("hipFree");
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = nullptr;
    const hipError_t e = done("hipHostMalloc");
    if (e != hipSuccess) return e;
    *p = std::calloc(n ? n : 1, 1);
    pinned[static_cast<char*>(*p)] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (pinned.erase(static_cast<char*>(p))) std::free(p);
    return done("hipHostFree");
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return done("hipHostGetDevicePointer");
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    std::memset(a, 0, sizeof(*a));
    a->type = inside(pinned, p) ? hipMemoryTypeHost : (inside(device, p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered);
    return done("hipPointerGetAttributes");
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return copy("hipMemcpy", d, s, n); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    return copy("hipMemcpyAsync", d, s, n);
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind,
                            hipStream_t) {
    const hipError_t e = done("hipMemcpy2DAsync");
    for (size_t k = 0; k < h && e == hipSuccess; ++k)
        std::memcpy(static_cast<char*>(d) + k * dp, static_cast<const char*>(s) + k * sp, w);
    return e;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
    std::memset(p, v, n);
    return done("hipMemsetAsync");
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = (size_t)1 << 40;
    return done("hipMemGetInfo");
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* scratch = std::calloc((size_t)64 << 20, 1);
    *p = scratch;
    return done("hipGetSymbolAddress");
}

// ---- device, streams, events, graphs
hipError_t hipSetDevice(int) { return done("hipSetDevice"); }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return done("hipGetDeviceCount");
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "stand-in");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    p->totalGlobalMem = (size_t)1 << 40;
    return done("hipGetDeviceProperties");
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 4;
    return done("hipOccupancyMaxActiveBlocksPerMultiprocessor");
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreate(hipStream_t* s) { return handle("hipStreamCreate", s); }
hipError_t hipStreamDestroy(hipStream_t) { return done("hipStreamDestroy"); }
hipError_t hipStreamSynchronize(hipStream_t) { return done("hipStreamSynchronize"); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return done("hipStreamWaitEvent"); }
hipError_t hipEventCreate(hipEvent_t* e) { return handle("hipEventCreate", e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle("hipEventCreateWithFlags", e); }
hipError_t hipEventDestroy(hipEvent_t) { return done("hipEventDestroy"); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return done("hipEventRecord"); }
hipError_t hipEventSynchronize(hipEvent_t) { return done("hipEventSynchronize"); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return done("hipEventElapsedTime");
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return done("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle("hipStreamEndCapture", g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* g, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return handle("hipGraphInstantiate", g);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return done("hipGraphLaunch"); }
hipError_t hipGraphDestroy(hipGraph_t) { return done("hipGraphDestroy"); }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return done("hipGraphExecDestroy"); }

// ---- launches
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return done("hipLaunchKernel"); }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = config.grid;
    *b = config.block;
    *lds = config.lds;
    *s = config.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
