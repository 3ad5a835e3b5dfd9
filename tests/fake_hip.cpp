// A stand-in for the HIP runtime in host memory, for CPU tests of the engine's
// host code: device buffers are host allocations, copies are real, kernels are
// not run.  Allocations and copies can be made to fail, and streams know the device
// they were made on.  Loaded with RTLD_GLOBAL before the
// engine library (or linked into a test program), it takes the place of every
// runtime call the engine makes after load.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <utility>

namespace {

std::mutex mu;
std::map<void*, size_t> bufs;
std::map<hipStream_t, int> streams;
thread_local int device = 0;
thread_local hipStream_t launch_stream = nullptr;
thread_local hipStreamCaptureMode capture_mode = hipStreamCaptureModeGlobal;
size_t live = 0, limit = ~(size_t)0;
int fail_copy = -1;       // copies to the host until one fails (-1: none does)
int slow_copy_ms = 0;     // what a copy to the host takes
long long misplaced = 0;  // kernels launched on a stream of another device than the current one
char symbol[1 << 22];

hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind kind) {
    if (kind == hipMemcpyDeviceToHost) {
        if (slow_copy_ms) std::this_thread::sleep_for(std::chrono::milliseconds(slow_copy_ms));
        std::lock_guard<std::mutex> g(mu);
        if (fail_copy >= 0 && fail_copy-- == 0) return hipErrorUnknown;
    }
    std::memcpy(d, s, n);
    return hipSuccess;
}

}  // namespace

extern "C" {

size_t fake_live_bytes() { return live; }
void fake_limit(size_t bytes) { limit = bytes; }  // hipMalloc fails beyond this many live bytes
void fake_fail_copy(int after) { fail_copy = after; }
void fake_slow_copy(int ms) { slow_copy_ms = ms; }
long long fake_misplaced() { return misplaced; }

hipError_t hipSetDevice(int d) {
    device = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, capture_mode);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> g(mu);
    if (live + n > limit) return hipErrorOutOfMemory;
    *p = std::calloc(1, n ? n : 1);
    if (!*p) return hipErrorOutOfMemory;
    bufs[*p] = n;
    live += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> g(mu);
    auto it = bufs.find(p);
    if (it == bufs.end()) return hipErrorInvalidValue;
    live -= it->second;
    std::free(p);
    bufs.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(1, n ? n : 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::mutex> g(mu);
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    streams[*s] = device;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::lock_guard<std::mutex> g(mu);
    streams.erase(s);
    std::free(reinterpret_cast<void*>(s));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(reinterpret_cast<void*>(e));
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
    std::memset(a, 0, sizeof(*a));
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = symbol;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) {
    launch_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = *b = dim3(1);
    *lds = 0;
    *s = launch_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) {
    std::lock_guard<std::mutex> g(mu);
    auto it = streams.find(s);
    if (it != streams.end() && it->second != device) ++misplaced;
    return hipSuccess;
}

}  // extern "C"
