// A HIP runtime without a device (test infrastructure), loaded in front of the real one by tests/test_conv_small_routes.py: kernels are noted by name and not run,
// allocations and waits are counted and refused while a stream is captured.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace
{
std::map<const void*, std::string>& names()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::string launched;
int allocations = 0;
bool captured = false;
char symbol[256];
}  // namespace

extern "C" {

void fake_capture(int on) { captured = on != 0; }
int fake_allocations() { return allocations; }
// names of the kernels launched since the last call, one a line
const char* fake_launched()
{
    static std::string out;
    out.swap(launched);
    launched.clear();
    return out.c_str();
}

void** __hipRegisterFatBinary(const void*)
{
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names()[host] = name; }

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = symbol; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return captured ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipMalloc(void** p, size_t)
{
    if (captured) return hipErrorStreamCaptureUnsupported;
    ++allocations;
    *p = malloc(1);
    return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
    *s = captured ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
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
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t)
{
    const auto it = names().find(f);
    launched += (it == names().end() ? std::string("?") : it->second) + "\n";
    return hipSuccess;
}
}
