// The HIP calls of the host-side sources, on the CPU: device and pinned memory are malloc's, a stream does its
// work at once, and an event is pending while `pending` is set.  Every call that a test looks at is in `calls`.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

static std::mutex fake_m;
static std::vector<std::string> fake_calls;
static std::atomic<bool> fake_pending{false};

static void call(const std::string& what)
{
    std::lock_guard<std::mutex> lock(fake_m);
    fake_calls.push_back(what);
}

static int count_calls(const std::string& what)
{
    std::lock_guard<std::mutex> lock(fake_m);
    int n = 0;
    for (const std::string& c : fake_calls) n += c == what;
    return n;
}

// Waits up to two seconds for the n-th call of that name.
static bool await_calls(const std::string& what, int n)
{
    for (int i = 0; i < 2000; ++i) {
        if (count_calls(what) >= n) return true;
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
    }
    return false;
}

#define CHECK(cond)                                                      \
    do {                                                                 \
        if (!(cond)) {                                                   \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #cond);      \
            std::_Exit(1);                                               \
        }                                                                \
    } while (0)

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
static hipError_t fake_last = hipSuccess;
hipError_t hipGetLastError()
{
    const hipError_t e = fake_last;
    fake_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = (hipStream_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    call("hipStreamSynchronize");
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t)
{
    call("hipStreamQuery");
    return fake_last = hipErrorNotReady;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned)
{
    call("hipStreamWaitEvent");
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return fake_pending ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n)
{
    call("hipMalloc");
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    call("hipHostMalloc");
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n)
{
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
}
