// A HIP runtime of two devices in host memory, as far as reading back needs it (test infrastructure): loaded in front of the real
// one by tests/test_read_back_route.py.  "Device memory" is host memory that the test has declared; the current device is the calling
// thread's; while a stream is captured a blocking copy is refused, whatever its size; an event belongs to the device that was current when it was made, and recording it from another is an error.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

namespace
{
struct Range { char* base; size_t bytes; hipMemoryType type; int device; };
std::mutex mu;
std::vector<Range> ranges;
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;   // of a launch
std::atomic<int> launches{0}, copies{0}, fail_launch{-1}, fail_pinned{0}, captured{0};
char symbol[256];

bool find(const void* p, Range* out)
{
    std::lock_guard<std::mutex> lock(mu);
    for (const Range& r : ranges)
        if ((const char*)p >= r.base && (const char*)p < r.base + r.bytes)
        {
            *out = r;
            return true;
        }
    return false;
}
void add(void* p, size_t bytes, hipMemoryType type, int device)
{
    std::lock_guard<std::mutex> lock(mu);
    ranges.push_back({(char*)p, bytes, type, device});
}
}  // namespace

extern "C" {

// kind 0: device memory, 1: pinned, 2: managed
void fake_declare(void* p, size_t bytes, int kind, int device)
{
    const hipMemoryType types[] = {hipMemoryTypeDevice, hipMemoryTypeHost, hipMemoryTypeManaged};
    add(p, bytes, types[kind], device);
}
void fake_reset(int launch_that_fails, int no_pinned_memory)
{
    launches = copies = 0;
    fail_launch = launch_that_fails;
    fail_pinned = no_pinned_memory;
}
void fake_capture(int on) { captured = on; }
int fake_launches() { return launches; }
int fake_copies() { return copies; }

hipError_t hipSetDevice(int d)
{
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    current = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = symbol; return hipSuccess; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    Range r;
    if (!find(p, &r)) return hipErrorInvalidValue;
    memset(a, 0, sizeof(*a));
    a->type = r.type;
    a->device = r.device;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* bytes, hipDeviceptr_t p)
{
    Range r;
    if (!find(p, &r)) return hipErrorInvalidValue;
    *base = r.base;
    *bytes = r.bytes;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned)
{
    if (fail_pinned) return hipErrorOutOfMemory;
    *p = malloc(bytes);
    add(*p, bytes, hipMemoryTypeHost, current);
    return hipSuccess;
}
hipError_t hipHostFree(void*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)new int(current);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return *(int*)e == current ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind)
{
    if (captured) return hipErrorStreamCaptureImplicit;
    copies += bytes > 0;
    if (!dst || !src) return hipErrorInvalidValue;
    memcpy(dst, src, bytes);
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error of the fake runtime"; }
const char* hipGetErrorName(hipError_t) { return "fake"; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st)
{
    *g = dim3(1);
    *b = dim3(1);
    *s = 0;
    *st = nullptr;
    return hipSuccess;
}
// The only kernel that reading back launches: (destination, source, bytes, wide), on the memory of the current device.
hipError_t hipLaunchKernel(const void*, dim3, dim3, void** args, size_t, hipStream_t)
{
    const int n = launches++;
    void* dst = *(void**)args[0];
    const void* src = *(const void**)args[1];
    Range r;
    if (n == fail_launch) return last = hipErrorLaunchFailure;
    if (!find(src, &r) || r.type != hipMemoryTypeDevice || r.device != current) return last = hipErrorIllegalAddress;
    memcpy(dst, src, *(size_t*)args[2]);
    return hipSuccess;
}
}
