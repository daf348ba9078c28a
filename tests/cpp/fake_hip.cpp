// A HIP runtime of host memory and no device, for tests of the library's host paths on the CPU: linked with the
// library's objects (bin/libmako_attn_fakehip.so), it records what a call allocates, frees and launches, in order, and
// runs no kernel. Device memory is malloc'd; a stream is any handle; the device has 256 compute units.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {

std::mutex mu;
std::string events;  // a line an event: alloc address bytes stream; free address; launch mangled-name grid stream
std::map<const void*, std::string> kernels;
std::map<void*, size_t> live;
std::set<hipStream_t> capturing;
size_t alloc_limit = SIZE_MAX;
void (*launch_hook)(const char* kernel) = nullptr;

thread_local struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} config;

__attribute__((format(printf, 1, 2))) void note(const char* fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    events += buf;
}

hipError_t allocate(void** p, size_t bytes, hipStream_t s)
{
    std::lock_guard<std::mutex> lock(mu);
    if (bytes > alloc_limit || posix_memalign(p, 4096, bytes ? bytes : 1))
        return hipErrorOutOfMemory;
    live[*p] = bytes;
    note("alloc %p %zu %p\n", *p, bytes, (void*)s);
    return hipSuccess;
}

hipError_t release(void* p)
{
    std::lock_guard<std::mutex> lock(mu);
    if (p && !live.erase(p))
        return hipErrorInvalidValue;
    note("free %p\n", p);
    std::free(p);
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- the tests' side ------------------------------------------------------------------------------------------------

// The events so far (valid until the next call here).
const char* fake_events()
{
    static std::string out;
    std::lock_guard<std::mutex> lock(mu);
    out = events;
    return out.c_str();
}

void fake_clear()
{
    std::lock_guard<std::mutex> lock(mu);
    events.clear();
}

void fake_capture(void* stream, int on)
{
    std::lock_guard<std::mutex> lock(mu);
    if (on)
        capturing.insert(static_cast<hipStream_t>(stream));
    else
        capturing.erase(static_cast<hipStream_t>(stream));
}

// Allocations of more than this many bytes fail.
void fake_alloc_limit(size_t bytes) { alloc_limit = bytes; }

// Called before each launch, on the launching thread (null: none).
void fake_launch_hook(void (*hook)(const char* kernel)) { launch_hook = hook; }

// ---- the library's side ---------------------------------------------------------------------------------------------

void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    std::lock_guard<std::mutex> lock(mu);
    kernels[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s)
{
    config = {grid, block, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s)
{
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t, hipStream_t s)
{
    std::string name;
    {
        std::lock_guard<std::mutex> lock(mu);
        name = kernels[f];
    }
    if (auto hook = launch_hook)
        hook(name.c_str());
    std::lock_guard<std::mutex> lock(mu);
    note("launch %s %u,%u,%u %p\n", name.c_str(), grid.x, grid.y, grid.z, (void*)s);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status)
{
    std::lock_guard<std::mutex> lock(mu);
    *status = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t s) { return allocate(p, bytes, s); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return release(p); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = std::malloc(4096);  // (never dereferenced)
    *p = scratch;
    return hipSuccess;
}

}  // extern "C"
