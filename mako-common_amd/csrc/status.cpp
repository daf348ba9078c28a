// The C ABI's error plumbing: a per-thread message for mako_last_error().
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <tuple>

#include "device.hpp"
#include "mako_attn.h"

namespace mako {

namespace {
thread_local std::string last_error;
thread_local int last_status = MAKO_OK;
}

int fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    last_error = buf;
    last_status = code;
    return code;
}

int ok()
{
    last_error.clear();
    last_status = MAKO_OK;
    return MAKO_OK;
}

int last_code() { return last_status; }

int check_launch(const char* what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return fail(MAKO_EHIP, "%s: launch failed: %s", what, hipGetErrorString(e));
    return ok();
}

uint32_t device_cus()
{
    static thread_local int dev_cached = -1;
    static thread_local uint32_t cus_cached = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return 0;
    if (dev != dev_cached) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            return 0;
        cus_cached = (uint32_t)cus;
        dev_cached = dev;
    }
    return cus_cached;
}

namespace {
// A stream's buffers, one a purpose. Entries stay (without memory) once made, so a reference outlives ws_mu.
struct StreamHeld {
    std::recursive_mutex turn;  // held by the call that uses the buffers
    struct {
        void* ptr = nullptr;
        std::atomic<size_t> bytes{0};  // (mako_attn_held_bytes reads it without the turn)
    } buf[kWsPurposes];
};
using StreamKey = std::tuple<int, hipStream_t, std::thread::id>;
std::mutex ws_mu;  // ws_all, not what its entries hold
std::map<StreamKey, StreamHeld> ws_all;

StreamKey stream_key(int dev, hipStream_t s)
{
    return {dev, s, s == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id()};
}
}  // namespace

void* Workspace::held(WorkspacePurpose which, size_t need, hipStream_t s) const
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return fail(MAKO_EHIP, "%s: no current device", what), nullptr;
    StreamHeld* all;
    {
        std::lock_guard<std::mutex> lock(ws_mu);
        all = &ws_all[stream_key(dev, s)];
    }
    if (!turn_.owns_lock())
        turn_ = std::unique_lock<std::recursive_mutex>(all->turn);
    auto& ws = all->buf[which];
    if (ws.bytes < need) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) != hipSuccess)
            (void)hipGetLastError();
        if (cap != hipStreamCaptureStatusNone)
            return fail(MAKO_EWORKSPACE,
                        "%s: the stream is capturing a graph and the library's workspace would grow to %zu bytes; "
                        "pass a workspace (the *_ws entry point) or make the call once before the capture",
                        what, need), nullptr;
        if (ws.ptr)
            (void)hipFreeAsync(ws.ptr, s);  // after the previous use on this stream
        ws.ptr = nullptr;
        ws.bytes = 0;
        if (hipMallocAsync(&ws.ptr, need, s) != hipSuccess) {
            (void)hipGetLastError();
            ws.ptr = nullptr;
            return fail(MAKO_EHIP, "%s: no device memory for a workspace of %zu bytes", what, need), nullptr;
        }
        ws.bytes = need;
    }
    return ws.ptr;
}

void* Workspace::get(size_t need, hipStream_t s) const
{
    if (!given)
        return held(purpose, need, s);
    if (bytes < need || (need && !ptr))
        return fail(MAKO_EWORKSPACE, "%s: a workspace of %zu bytes, the call needs %zu", what, bytes, need), nullptr;
    return ptr;
}

void* Workspace::try_get(WorkspacePurpose optional, size_t need, hipStream_t s) const
{
    if (given)
        return bytes >= need && reinterpret_cast<uintptr_t>(ptr) % 16 == 0 ? ptr : nullptr;
    if (s == hipStreamPerThread)
        return nullptr;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess)
        (void)hipGetLastError();
    return cap == hipStreamCaptureStatusNone ? held(optional, need, s) : nullptr;
}

Workspace Workspace::at(size_t offset) const
{
    if (!given)
        return library_workspace(purpose, what);
    return offset <= bytes ? caller_workspace(static_cast<char*>(ptr) + offset, bytes - offset, what)
                           : caller_workspace(nullptr, 0, what);
}

}  // namespace mako

extern "C" int mako_attn_abi_version(void) { return MAKO_ATTN_ABI_VERSION; }

extern "C" int mako_attn_release(void* stream)
{
    using namespace mako;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return fail(MAKO_EHIP, "release: no current device");
    StreamHeld* all = nullptr;
    {
        std::lock_guard<std::mutex> lock(ws_mu);
        const auto it = ws_all.find(stream_key(dev, s));
        if (it != ws_all.end())
            all = &it->second;
    }
    std::unique_lock<std::recursive_mutex> turn;
    if (all)
        turn = std::unique_lock<std::recursive_mutex>(all->turn);
    if (hipStreamSynchronize(s) != hipSuccess)
        return fail(MAKO_EHIP, "release: %s", hipGetErrorString(hipGetLastError()));
    if (all)
        for (auto& ws : all->buf) {
            if (ws.ptr && hipFree(ws.ptr) != hipSuccess)
                return fail(MAKO_EHIP, "release: %s", hipGetErrorString(hipGetLastError()));
            ws.ptr = nullptr;
            ws.bytes = 0;
        }
    return ok();
}

extern "C" size_t mako_attn_held_bytes(void)
{
    using namespace mako;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return 0;
    std::lock_guard<std::mutex> lock(ws_mu);
    size_t n = 0;
    for (const auto& kv : ws_all)
        if (std::get<0>(kv.first) == dev)
            for (const auto& ws : kv.second.buf)
                n += ws.bytes;
    return n;
}

extern "C" const char* mako_last_error(void) { return mako::last_error.c_str(); }
