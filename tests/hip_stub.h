// hip_stub.h — a HIP runtime for host checks of libvolprim.so, which a check
// program defines itself, so that the library's calls reach it instead of
// libamdhip64: device memory is host memory (zeroed, counted, limited), work
// on a stream is queued and done when something waits for it, kernels do
// nothing but for the two that move words, and chosen calls fail.
#pragma once

#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace stub {

inline std::recursive_mutex mu;  // of everything below
inline std::deque<std::function<void()>> queue;  // of every stream
inline std::map<void*, size_t> device_mem, pinned_mem;
inline size_t used = 0, limit = ~size_t(0);  // device bytes
inline int device = 0;                       // current device
// kernels by their host functions (registered before this program's own variables are initialised)
inline std::map<const void*, std::string>& kernels() {
    static auto* m = new std::map<const void*, std::string>();
    return *m;
}
// called for every launch (kernel, workgroup; its arguments are in launch_args);
// an error is its result
inline void** launch_args = nullptr;
inline std::function<hipError_t(const std::string&, dim3)> on_launch;
// called for every queued copy and recorded event; an error is its result
inline std::function<hipError_t()> on_copy, on_record;
inline hipError_t last = hipSuccess;
inline bool replayed = false;  // a graph ran: its next count of paths is complete

struct Stream {
    int device;
};

inline hipError_t keep(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
inline void drain() {
    while (!queue.empty()) {
        queue.front()();
        queue.pop_front();
    }
}
inline void check(bool ok, const char* what) {
    if (ok) return;
    std::printf("FAILED: %s\n", what);
    std::fflush(stdout);
    std::_Exit(1);
}

}  // namespace stub

#define STUB_LOCK std::lock_guard<std::recursive_mutex> lk(stub::mu)

extern "C" {

hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipSetDevice(int d) { return stub::device = d, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    STUB_LOCK;
    if (stub::used + bytes > stub::limit) return stub::keep(hipErrorOutOfMemory);
    *p = std::calloc(1, bytes ? bytes : 1);
    stub::device_mem[*p] = bytes;
    stub::used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    STUB_LOCK;
    stub::drain();
    if (!p) return hipSuccess;
    stub::check(stub::device_mem.count(p) == 1, "hipFree of memory that is not allocated");
    stub::used -= stub::device_mem[p];
    stub::device_mem.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t) { return hipMalloc(p, bytes); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return hipFree(p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) {
    STUB_LOCK;
    *p = std::calloc(1, bytes ? bytes : 1);
    stub::pinned_mem[*p] = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    STUB_LOCK;
    stub::drain();
    stub::pinned_mem.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    STUB_LOCK;
    std::memset(a, 0, sizeof(*a));
    a->type = stub::pinned_mem.count(const_cast<void*>(p)) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t) {
    STUB_LOCK;
    if (stub::on_copy) {
        const hipError_t e = stub::on_copy();
        if (e != hipSuccess) return stub::keep(e);
    }
    if (stub::replayed && kind == hipMemcpyDeviceToHost && bytes == sizeof(unsigned long long)) {
        stub::queue.push_back([=] { *static_cast<unsigned long long*>(dst) = ~0ull; });
        return hipSuccess;
    }
    stub::queue.push_back([=] { std::memcpy(dst, src, bytes); });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t bytes, hipStream_t) {
    STUB_LOCK;
    stub::queue.push_back([=] { std::memset(p, v, bytes); });
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = reinterpret_cast<hipStream_t>(new stub::Stream{stub::device});
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { return hipStreamCreate(s); }
hipError_t hipExtStreamCreateWithCUMask(hipStream_t* s, uint32_t, const uint32_t*) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) {
    delete reinterpret_cast<stub::Stream*>(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    STUB_LOCK;
    stub::drain();
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(new int(0)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<int*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
    STUB_LOCK;
    return stub::on_record ? stub::keep(stub::on_record()) : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventQuery(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    return *g = reinterpret_cast<hipGraph_t>(new int(0)), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *x = reinterpret_cast<hipGraphExec_t>(new int(0)), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete reinterpret_cast<int*>(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    delete reinterpret_cast<int*>(x);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    STUB_LOCK;
    stub::replayed = true;
    return stub::on_launch ? stub::keep(stub::on_launch("graph", dim3(1))) : hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = stub::last;
    stub::last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
// 16 wavefronts to a compute unit
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int block, size_t) {
    return *n = 1024 / block, hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static std::vector<char> scratch(size_t(136) << 20);
    return *p = scratch.data(), hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return new void*(nullptr); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, void*, void*,
                           int*) {
    stub::kernels()[host] = name;
}
static thread_local dim3 stub_grid, stub_block;
static thread_local size_t stub_lds;
static thread_local hipStream_t stub_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    stub_grid = g, stub_block = b, stub_lds = lds, stub_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = stub_grid, *b = stub_block, *lds = stub_lds, *s = stub_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3, dim3 block, void** args, size_t, hipStream_t s) {
    STUB_LOCK;
    const std::string& name = stub::kernels()[host];
    if (s && reinterpret_cast<stub::Stream*>(s)->device != stub::device) return stub::keep(hipErrorInvalidHandle);
    stub::launch_args = args;
    if (stub::on_launch) {
        const hipError_t e = stub::on_launch(name, block);
        if (e != hipSuccess) return stub::keep(e);
    }
    if (name.find("k_copy_parts") != std::string::npos) {
        struct Parts {  // CopyParts
            const uint32_t* src[4];
            uint32_t* dst[4];
            uint32_t words[4];
        } c = *static_cast<Parts*>(args[0]);
        stub::queue.push_back([=] {
            for (int k = 0; k < 4; ++k) std::memcpy(c.dst[k], c.src[k], 4 * size_t(c.words[k]));
        });
    }
    return hipSuccess;
}

}  // extern "C"
