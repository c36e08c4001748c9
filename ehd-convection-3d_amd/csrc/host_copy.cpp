// host_copy.cpp -- see host_copy.h.
//
// A plain hipMemcpy of fields into an array that the caller has just
// allocated runs at 4 GB/s (single-threaded page faults and pinning), twice
// the time of the steps between two outputs.  Here the device copies 2 MB
// pieces into pinned slots (56 GB/s) while worker threads move them on into
// the caller's pages, whose first touch is what costs; floats cross the bus as
// floats and are widened by the workers.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "box.h"

namespace ehd {
namespace {

constexpr size_t kSlot = (size_t)2 << 20;   // bytes of a slot, on the device's side
constexpr int kSlots = 8;
constexpr int kWorkers = 6;
constexpr size_t kAlone = (size_t)1 << 20;  // up to this much the calling thread moves by itself

struct Staging {
    char* mem = nullptr;             // kSlots slots, then kMaxMean doubles
    hipEvent_t ev[kSlots] = {};
    int device = -1;

    double* mean() const { return (double*)(mem + kSlots * kSlot); }
    // with dev current: an event can only be recorded on a stream of its own device
    bool make(int dev)
    {
        device = dev;
        if (hipHostMalloc((void**)&mem, kSlots * kSlot + kMaxMean * sizeof(double), hipHostMallocDefault) != hipSuccess) {
            mem = nullptr;
            return false;
        }
        for (hipEvent_t& e : ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return false;
            }
        return true;
    }
    ~Staging()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex g_mu;
// A buffer costs milliseconds to allocate and to free: eight are kept (128 MB
// pinned at most), one for each device of a node or each of as many readers.
constexpr int kKept = 8;
Staging* g_kept[kKept] = {};
long long g_owners = 0;

// a staging buffer of the stream's device (the calling thread's may be another)
// for one call, given back (or freed, when kKept are kept already or no owner is
// left) at the end of it
struct Lease {
    Staging* s = nullptr;
    explicit Lease(hipStream_t st)
    {
        int dev = -1, current = -1;
        if (hipStreamGetDevice(st, &dev) != hipSuccess || hipGetDevice(&current) != hipSuccess) {
            (void)hipGetLastError();   // the copies go without staging: the next check of a launch must not find it
            return;
        }
        {
            std::lock_guard<std::mutex> lk(g_mu);
            for (Staging*& k : g_kept)
                if (k && k->device == dev) {
                    s = k;
                    k = nullptr;
                    return;
                }
        }
        s = new (std::nothrow) Staging();
        if (current != dev && hipSetDevice(dev) != hipSuccess) dev = -1;
        if (s && (dev < 0 || !s->make(dev))) {
            delete s;
            s = nullptr;
            (void)hipGetLastError();
        }
        if (current != dev && dev >= 0) (void)hipSetDevice(current);
    }
    ~Lease()
    {
        if (!s) return;
        {
            std::lock_guard<std::mutex> lk(g_mu);
            if (g_owners > 0)
                for (Staging*& k : g_kept)
                    if (!k) {
                        k = s;
                        return;
                    }
        }
        delete s;
    }
};

size_t width(const HostCopy& c) { return c.kind == HostCopy::kDouble ? sizeof(double) : sizeof(float); }

// elements i0 .. i0 + n of array c, from a slot to the caller's memory
void deliver(const HostCopy& c, const void* slot, size_t i0, size_t n, const double* mean)
{
    if (c.kind == HostCopy::kFloat) {
        std::memcpy((float*)c.host + i0, slot, n * sizeof(float));
    } else if (c.kind == HostCopy::kDouble) {
        std::memcpy((double*)c.host + i0, slot, n * sizeof(double));
    } else {
        const float* src = (const float*)slot;
        double* dst = (double*)c.host + i0;
        if (c.kind == HostCopy::kWiden) {
            for (size_t i = 0; i < n; ++i) dst[i] = (double)src[i];
        } else {
            for (size_t i = 0; i < n;) {
                const size_t z = (i0 + i) / c.plane, e = std::min(n, (z + 1) * c.plane - i0);
                const double m = mean[z];
                for (; i < e; ++i) dst[i] = (double)src[i] + m;
            }
        }
    }
}

struct Piece {
    int array;
    size_t i0, n;
};

// Worker threads that take the pieces of one call in order.  The calling
// thread alone talks to the device: it raises `ready` when a piece may be
// taken and waits for a piece to be done before it reuses its slot.  A call
// lasts milliseconds and its pieces tens of microseconds, less than it takes
// to put a thread to sleep and wake it: all sides spin (and yield).
class Crew {
public:
    template <class F>
    Crew(int pieces, const F& work) : done_(new std::atomic<char>[pieces])
    {
        for (int k = 0; k < pieces; ++k) done_[k] = 0;
        auto run = [this, pieces, work] {
            for (int k; (k = next_.fetch_add(1)) < pieces;) {
                while (k >= ready_.load(std::memory_order_acquire)) {
                    if (stop_.load(std::memory_order_relaxed)) return;
                    std::this_thread::yield();
                }
                work(k);
                done_[k].store(1, std::memory_order_release);
            }
        };
        try {
            for (int t = 0; t < std::min(kWorkers, pieces); ++t) crew_.emplace_back(run);
        } catch (...) {   // fewer threads than asked for; with none the caller does the work
        }
    }
    ~Crew()
    {
        stop_ = true;
        for (std::thread& t : crew_) t.join();
    }
    bool empty() const { return crew_.empty(); }
    void raise(int ready) { ready_.store(ready, std::memory_order_release); }
    void wait(int k)
    {
        while (!done_[k].load(std::memory_order_acquire)) std::this_thread::yield();
    }

private:
    std::unique_ptr<std::atomic<char>[]> done_;
    std::vector<std::thread> crew_;
    std::atomic<int> next_{0}, ready_{0};
    std::atomic<bool> stop_{false};
};

// On every way out that is not a return of EHD_OK, no copy on the stream
// outlives the memory that it writes: declared after all of that.
struct Drain {
    hipStream_t st;
    bool done = false;
    ~Drain()
    {
        if (!done) (void)hipStreamSynchronize(st);
    }
};

// without staging memory or threads: as the runtime does it
int download_plain(const HostCopy* c, int count, hipStream_t st)
{
    std::vector<float> f;
    std::vector<double> mean;
    Drain drain{st};
    for (int a = 0; a < count; ++a) {
        const bool raw = c[a].kind == HostCopy::kFloat || c[a].kind == HostCopy::kDouble;
        void* to = c[a].host;
        if (!raw) {
            f.resize(c[a].n);
            to = f.data();
        }
        HIPCHK(hipMemcpyAsync(to, c[a].dev, c[a].n * width(c[a]), hipMemcpyDeviceToHost, st));
        if (c[a].kind == HostCopy::kWidenAddMean) {
            mean.resize(c[a].nmean);
            HIPCHK(hipMemcpyAsync(mean.data(), c[a].mean, c[a].nmean * sizeof(double), hipMemcpyDeviceToHost, st));
        }
        HIPCHK(hipStreamSynchronize(st));
        if (!raw) deliver(c[a], f.data(), 0, c[a].n, mean.data());
    }
    drain.done = true;
    return EHD_OK;
}

int download_staged(const HostCopy* c, int count, hipStream_t st, Staging& S)
{
    Drain drain{st};
    std::vector<Piece> pieces;
    size_t total = 0;
    for (int a = 0; a < count; ++a) {
        const size_t step = kSlot / width(c[a]);
        for (size_t i0 = 0; i0 < c[a].n; i0 += step) pieces.push_back({a, i0, std::min(step, c[a].n - i0)});
        total += c[a].n * width(c[a]);
        if (c[a].kind == HostCopy::kWidenAddMean)   // ahead of every piece on the stream
            HIPCHK(hipMemcpyAsync(S.mean(), c[a].mean, c[a].nmean * sizeof(double), hipMemcpyDeviceToHost, st));
    }
    const int np = (int)pieces.size();
    auto fetch = [&](int k, char* slot) {
        const Piece& p = pieces[k];
        const size_t w = width(c[p.array]);
        return hipMemcpyAsync(slot, (const char*)c[p.array].dev + p.i0 * w, p.n * w, hipMemcpyDeviceToHost, st);
    };
    auto move = [&](int k, const char* slot) {
        deliver(c[pieces[k].array], slot, pieces[k].i0, pieces[k].n, S.mean());
    };
    if (total <= kAlone) {
        // everything behind one wait
        char* at = S.mem;
        for (int k = 0; k < np; ++k) {
            HIPCHK(fetch(k, at));
            at += (pieces[k].n * width(c[pieces[k].array]) + 63) & ~(size_t)63;
        }
        HIPCHK(hipStreamSynchronize(st));
        at = S.mem;
        for (int k = 0; k < np; ++k) {
            move(k, at);
            at += (pieces[k].n * width(c[pieces[k].array]) + 63) & ~(size_t)63;
        }
        drain.done = true;
        return EHD_OK;
    }
    auto slot = [&](int k) { return S.mem + (size_t)(k % kSlots) * kSlot; };
    auto send = [&](int k) {
        const hipError_t e = fetch(k, slot(k));
        return e == hipSuccess ? hipEventRecord(S.ev[k % kSlots], st) : e;
    };
    hipError_t e = hipSuccess;
    int sent = 0;
    while (sent < std::min(np, kSlots) && e == hipSuccess) e = send(sent++);
    // the work queued before may take long: no thread is started until the first piece is here
    if (e == hipSuccess) e = hipEventSynchronize(S.ev[0]);
    if (e == hipSuccess) {
        Crew crew(np, [&](int k) { move(k, slot(k)); });
        for (int k = 0; k < np && e == hipSuccess; ++k) {
            e = hipEventSynchronize(S.ev[k % kSlots]);
            if (e != hipSuccess) break;
            if (crew.empty()) move(k, slot(k));
            else crew.raise(k + 1);
            // refill the slots half the ring behind, which are most likely free
            const int old = k + 1 - kSlots / 2;
            if (old >= 0 && sent < np && sent == old + kSlots) {
                if (!crew.empty()) crew.wait(old);
                e = send(sent++);
            }
        }
        // Everything has arrived.  The stream is waited for too, which has a thread
        // of the runtime finish the copies' commands, here beside the last
        // deliveries; left undone, that was on the bill of whatever the owner of the
        // stream did next (ehd_read_fields).
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e == hipSuccess && !crew.empty())
            for (int k = std::max(0, np - kSlots); k < np; ++k) crew.wait(k);
    }
    if (e != hipSuccess) return set_error(EHD_EHIP, "device to host copy failed: %s", hipGetErrorString(e));
    drain.done = true;
    return EHD_OK;
}

}  // namespace

int download(const HostCopy* c, int count, hipStream_t st)
{
    try {
        Lease lease(st);
        return lease.s ? download_staged(c, count, st, *lease.s) : download_plain(c, count, st);
    } catch (const std::bad_alloc&) {
        return set_error(EHD_ENOMEM, "host allocation failed");
    }
}

void staging_retain()
{
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_owners;
}

void staging_release()
{
    Staging* drop[kKept] = {};
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (--g_owners == 0)
            for (int i = 0; i < kKept; ++i) std::swap(drop[i], g_kept[i]);
    }
    for (Staging* s : drop) delete s;
}

}  // namespace ehd
