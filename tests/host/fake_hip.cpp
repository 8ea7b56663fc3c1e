#include "fake_hip.h"

#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>

namespace fake_hip {
long launches = 0, other_device = 0, out_of_range = 0;
thread_local int inside = 0;
}

namespace {

struct State {  // (in a function: kernels are registered by other files' static constructors)
    std::recursive_mutex mu;
    std::map<uintptr_t, size_t> device, pinned;  // base -> bytes
    std::map<const void*, std::string> kernels;
    std::map<const void*, void*> symbols;
    std::deque<std::function<void()>> queue;
    std::vector<std::pair<std::string, dim3>> enqueued;  // kernels, mangled, and their grids
    bool capturing = false;
    long launch_fails = 0, copy_fails = 0;
    bool pinned_fails = false;
};
State& st() {
    static State* s = new State;
    return *s;
}
struct Lock {
    std::lock_guard<std::recursive_mutex> lk{st().mu};
    Lock() { fake_hip::inside++; }
    ~Lock() { fake_hip::inside--; }
};
thread_local hipError_t last = hipSuccess;
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config config;
thread_local int current = 0;  // the thread's GPU; the streams' handles are one past theirs

hipError_t done(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}

// The allocation that holds p, or null.
const std::pair<const uintptr_t, size_t>* holder(const std::map<uintptr_t, size_t>& of, const void* p) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    auto it = of.upper_bound(a);
    if (it == of.begin()) return nullptr;
    --it;
    return a < it->first + it->second ? &*it : nullptr;
}
bool covers(const void* p, size_t n) {
    for (const auto* of : {&st().device, &st().pinned})
        if (const auto* h = holder(*of, p)) return reinterpret_cast<uintptr_t>(p) + n <= h->first + h->second;
    return false;
}

bool due(long& n) { return n > 0 && --n == 0; }

void drain() {
    Lock lk;
    while (!st().queue.empty()) {
        st().queue.front()();
        st().queue.pop_front();
    }
}

void enqueue(std::function<void()> f) {
    if (!st().capturing) st().queue.push_back(std::move(f));
}

hipError_t launch(const void* f, dim3 grid, void** args, hipStream_t stream) {
    Lock lk;
    if (reinterpret_cast<uintptr_t>(stream) != (uintptr_t)current + 1) fake_hip::other_device++;
    if (due(st().launch_fails)) return done(hipErrorLaunchFailure);
    fake_hip::launches++;
    st().enqueued.push_back({st().kernels[f], grid});
    if (st().kernels[f].find("rmsnorm_quantize_kernel") != std::string::npos) {  // (x, shares, their stride, weight, quants, scales, dim, ..)
        const size_t elements = (size_t)grid.x * *static_cast<uint32_t*>(args[6]);
        if (!covers(*static_cast<void**>(args[4]), elements) || !covers(*static_cast<void**>(args[5]), elements / 32 * sizeof(float))) fake_hip::out_of_range++;
    }
    if (st().kernels[f].find("stage_copy_kernel") == std::string::npos) {
        enqueue([] {});
        return hipSuccess;
    }
    const void* src = *static_cast<const void**>(args[0]);
    void* dst = *static_cast<void**>(args[1]);
    const uint32_t n = *static_cast<uint32_t*>(args[2]);
    enqueue([=] {
        if (!covers(src, n) || !covers(dst, n)) fake_hip::out_of_range++;
        else std::memcpy(dst, src, n);
    });
    return hipSuccess;
}

hipError_t allocate(std::map<uintptr_t, size_t>& in, void** p, size_t n) {
    Lock lk;
    if (posix_memalign(p, 256, (n + 255) / 256 * 256) != 0) return done(hipErrorOutOfMemory);
    in[reinterpret_cast<uintptr_t>(*p)] = n;
    return hipSuccess;
}
hipError_t release(std::map<uintptr_t, size_t>& in, void* p) {
    if (!p) return hipSuccess;
    drain();
    Lock lk;
    if (in.erase(reinterpret_cast<uintptr_t>(p)) == 0) return done(hipErrorInvalidValue);
    std::free(p);
    return hipSuccess;
}

template <typename T>
T handle() {
    static char h[64];
    return reinterpret_cast<T>(h);
}

}  // namespace

namespace fake_hip {
size_t pending() {
    Lock lk;
    return st().queue.size();
}
size_t allocations() {
    Lock lk;
    return st().device.size();
}
std::vector<std::string> kernels() {
    Lock lk;
    std::vector<std::string> names;
    for (const auto& [mangled, grid] : st().enqueued) {
        char* const plain = abi::__cxa_demangle(mangled.c_str(), nullptr, nullptr, nullptr);
        names.push_back((plain ? plain : mangled) + (" (" + std::to_string(grid.x) + " x " + std::to_string(grid.y) + ")"));
        std::free(plain);
    }
    st().enqueued.clear();
    return names;
}
void fail_launch(long n) {
    Lock lk;
    st().launch_fails = n;
}
void fail_copy(long n) {
    Lock lk;
    st().copy_fails = n;
}
void fail_pinned(bool on) {
    Lock lk;
    st().pinned_fails = on;
}
}  // namespace fake_hip

extern "C" {

void** __hipRegisterFatBinary(const void*) { return handle<void**>(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { st().kernels[host] = name; }
void __hipRegisterVar(void**, void* host, char*, char*, int, size_t size, int, int) {
    void* p = nullptr;
    if (allocate(st().pinned, &p, size) == hipSuccess) st().symbols[host] = p;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    config = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = config.grid, *block = config.block, *shared = config.shared, *stream = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s) { return launch(f, grid, args, s); }
hipError_t hipExtLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s, hipEvent_t, hipEvent_t, int) { return launch(f, grid, args, s); }

hipError_t hipGetDeviceCount(int* n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    current = d;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = 1ull << 30;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "an error of the test's"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    *p = st().symbols[symbol];
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) { return allocate(st().device, p, n); }
hipError_t hipFree(void* p) { return release(st().device, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return st().pinned_fails ? done(hipErrorOutOfMemory) : allocate(st().pinned, p, n); }
hipError_t hipHostFree(void* p) { return release(st().pinned, p); }
// As the runtime does: a range that starts in an allocation has to end in it; two addresses it does not know are a copy on the host.
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    Lock lk;
    if (due(st().copy_fails)) return done(hipErrorLaunchFailure);
    for (const void* p : {static_cast<const void*>(dst), src})
        if ((holder(st().device, p) || holder(st().pinned, p)) && !covers(p, n)) return done(hipErrorInvalidValue);
    enqueue([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    Lock lk;
    for (const auto* of : {&st().device, &st().pinned})
        if (const auto* h = holder(*of, p)) {
            if (base) *base = reinterpret_cast<hipDeviceptr_t>(h->first);
            if (size) *size = h->second;
            return hipSuccess;
        }
    return done(hipErrorNotFound);
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    Lock lk;
    std::memset(a, 0, sizeof *a);
    a->type = holder(st().device, p) ? hipMemoryTypeDevice : (holder(st().pinned, p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered);
    if (a->type == hipMemoryTypeUnregistered) a->device = -2;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>((uintptr_t)current + 1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    drain();
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    st().capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    st().capturing = false;
    *g = handle<hipGraph_t>();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = handle<hipGraphExec_t>();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    Lock lk;
    enqueue([] {});
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) {
    *e = handle<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    drain();
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}

}  // extern "C"
