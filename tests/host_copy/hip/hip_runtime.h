// hip_runtime.h -- a stand-in for the HIP runtime on the CPU, for the tests of
// host code that queues copies: device memory is host memory, a stream keeps
// its commands until something waits for them, and a call can be told to fail.
#pragma once

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>

#define __host__
#define __device__

typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400;
constexpr int HIP_VERSION = 70200000;   // the runtime that the code is built for
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipStreamNonBlocking = 1;

namespace fake {

struct Stream {
    int device = 0;
    long queued = 0, run = 0;      // commands so far, and those of them that have run
    long waited = 0;               // commands that a wait for the whole stream has covered
    std::deque<std::function<void()>> todo;

    void drain(long upto)
    {
        while (run < upto) {
            todo.front()();
            todo.pop_front();
            ++run;
        }
    }
};

struct Event {
    int device = 0;
    Stream* stream = nullptr;
    long at = 0;
};

inline std::recursive_mutex mu;
inline std::map<std::string, long> calls;     // how often a call was made
inline std::string failing;                   // this call fails
inline long failing_from = 0;                 // from this call of it on (counting from 1)
inline int version = HIP_VERSION;             // of the runtime that is there
inline thread_local int current = 0;          // current device
inline thread_local hipError_t last = hipSuccess;
inline std::map<char*, size_t> pinned;        // pinned allocations alive
inline std::map<char*, long> targets;         // where the copies that have not run yet will write
inline long freed_early = 0;                  // pinned allocations freed ahead of such a copy

// counts the call; an error to return, which also stays in the thread
inline hipError_t enter(const char* name, hipError_t error = hipErrorInvalidValue)
{
    const long n = ++calls[name];
    if (failing == name && n >= failing_from) return last = error;
    return hipSuccess;
}

inline void fail(const std::string& name, long from)
{
    failing = name;
    failing_from = calls[name] + from;
}

}  // namespace fake

typedef fake::Stream* hipStream_t;
typedef fake::Event* hipEvent_t;

inline const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "an error"; }

inline hipError_t hipGetLastError()
{
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}

inline hipError_t hipGetDevice(int* d)
{
    *d = fake::current;
    return hipSuccess;
}

inline hipError_t hipSetDevice(int d)
{
    fake::current = d;
    return hipSuccess;
}

inline hipError_t hipStreamGetDevice(hipStream_t s, int* d)
{
    *d = s->device;
    return hipSuccess;
}

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t e = fake::enter("hipHostMalloc", hipErrorOutOfMemory)) return e;
    *p = std::malloc(n);
    fake::pinned[(char*)*p] = n;
    return hipSuccess;
}

inline hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    for (const auto& t : fake::targets)
        if (t.second > 0 && t.first >= (char*)p && t.first < (char*)p + fake::pinned[(char*)p]) {
            ++fake::freed_early;
            return hipSuccess;   // kept, so that the copy has a target
        }
    fake::pinned.erase((char*)p);
    std::free(p);
    return hipSuccess;
}

inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t r = fake::enter("hipEventCreateWithFlags", hipErrorOutOfMemory)) return r;
    *e = new fake::Event{fake::current};
    return hipSuccess;
}

inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}

inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t r = fake::enter("hipEventRecord")) return r;
    if (e->device != s->device) return fake::last = hipErrorInvalidHandle;
    s->todo.push_back([] {});
    e->stream = s;
    e->at = ++s->queued;
    return hipSuccess;
}

inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t r = fake::enter("hipEventSynchronize")) return r;
    if (e->stream) e->stream->drain(e->at);
    return hipSuccess;
}

inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t r = fake::enter("hipStreamSynchronize")) return r;
    s->drain(s->queued);
    s->waited = s->queued;
    return hipSuccess;
}

inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lk(fake::mu);
    if (const hipError_t r = fake::enter("hipMemcpyAsync")) return r;
    ++fake::targets[(char*)to];
    s->todo.push_back([=] {
        std::memcpy(to, from, n);
        --fake::targets[(char*)to];
    });
    ++s->queued;
    return hipSuccess;
}

// ---- what a batch uses beside copies: plain memory, events without time, graphs that only count ----

struct fakeGraph {
};
typedef fakeGraph* hipGraph_t;
typedef fakeGraph* hipGraphExec_t;

inline hipError_t hipRuntimeGetVersion(int* v)
{
    *v = fake::version;
    return fake::enter("hipRuntimeGetVersion");
}

template <class T>
hipError_t hipMalloc(T** p, size_t n)
{
    *p = (T*)std::malloc(n);
    return hipSuccess;
}

inline hipError_t hipFree(void* p)
{
    std::free(p);
    return hipSuccess;
}

inline hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind)
{
    std::memcpy(to, from, n);
    return hipSuccess;
}

inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = new fake::Stream;
    return hipSuccess;
}

inline hipError_t hipStreamDestroy(hipStream_t s)
{
    delete s;
    return hipSuccess;
}

inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }

inline hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }

inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}

inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return fake::enter("hipStreamBeginCapture"); }

inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = new fakeGraph;
    return hipSuccess;
}

inline hipError_t hipGraphDestroy(hipGraph_t g)
{
    delete g;
    return hipSuccess;
}

inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, char*, size_t)
{
    *e = new fakeGraph;
    return hipSuccess;
}

inline hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
    delete e;
    return hipSuccess;
}

inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return fake::enter("hipGraphLaunch"); }
