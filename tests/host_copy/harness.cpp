// harness.cpp -- drives host_copy.cpp on the stand-in runtime beside this
// file; tests/test_host_copy.py builds it and runs one scenario per call.
// Prints "ok" at the end.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>

#include "../../ehd-convection-3d_amd/csrc/box.h"
#include "../../ehd-convection-3d_amd/csrc/host_copy.h"

#define CHECK(c)                                                                         \
    do {                                                                                 \
        if (!(c)) {                                                                      \
            std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c);          \
            std::exit(3);                                                                \
        }                                                                                \
    } while (0)

// an array allocation of this size runs out of memory
static size_t g_no_memory = 0;
void* operator new[](size_t n)
{
    if (n == g_no_memory) throw std::bad_alloc();
    void* p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete[](void* p, size_t) noexcept { std::free(p); }

using namespace ehd;

namespace {

constexpr size_t kPiece = ((size_t)2 << 20) / 4;   // floats of a piece

// one field of n floats, another with the mean of its planes, and their copies
struct Fields {
    std::vector<float> a, b;
    std::vector<double> mean, wide, full;
    HostCopy c[2];

    explicit Fields(size_t n, size_t planes = 4) : a(n), b(n), mean(planes), wide(n, -1.0), full(n, -1.0)
    {
        for (size_t i = 0; i < n; ++i) {
            a[i] = (float)(i % 1013) + 0.5f;
            b[i] = (float)(i % 911) - 0.25f;
        }
        for (size_t z = 0; z < planes; ++z) mean[z] = 1e-9 * (double)(z + 1);
        c[0] = HostCopy{HostCopy::kWiden, wide.data(), a.data(), n};
        c[1] = HostCopy{HostCopy::kWidenAddMean, full.data(), b.data(), n, mean.data(), planes, n / planes};
    }
    bool right() const
    {
        for (size_t i = 0; i < a.size(); ++i)
            if (wide[i] != (double)a[i] || full[i] != (double)b[i] + mean[i / (a.size() / mean.size())]) return false;
        return true;
    }
};

const size_t kSizes[] = {400, 6 * kPiece - 400};   // behind one wait; through the ring of 8, 12 pieces

void exact()
{
    fake::Stream st;
    for (size_t n : kSizes) {
        Fields f(n);
        CHECK(download(f.c, 2, &st) == EHD_OK && f.right());
    }
}

// Whatever call of the copies fails, none of them is left on the stream when
// the staging memory is given back, here (no owner is counted in) freed.
void failing(const std::string& call)
{
    for (size_t n : kSizes)
        for (long k = 1; k <= 30; ++k) {
            Fields f(n), g(n);
            fake::Stream st, other;
            fake::fail(call, k);
            const int rc = download(f.c, 2, &st);
            fake::failing.clear();
            CHECK(st.run == st.queued && fake::freed_early == 0);
            CHECK(rc != EHD_OK || f.right());
            CHECK(download(g.c, 2, &other) == EHD_OK && g.right());
        }
}

void no_memory()
{
    fake::Stream st, other;
    Fields f(kSizes[1]), g(kSizes[1]);
    g_no_memory = 12;   // the table of its pieces
    CHECK(download(f.c, 2, &st) == EHD_ENOMEM);
    g_no_memory = 0;
    CHECK(st.run == st.queued && fake::freed_early == 0);
    CHECK(download(g.c, 2, &other) == EHD_OK && g.right());
}

// Without staging memory the copies go the plain way, and the failure that the
// call got over is not found by the next check of the thread's last error.
void no_staging(const std::string& call)
{
    for (size_t n : kSizes)
        for (long k = 1; k <= (call == "hipHostMalloc" ? 1 : 8); ++k) {
            Fields f(n);
            fake::Stream st;
            fake::fail(call, k);
            CHECK(download(f.c, 2, &st) == EHD_OK && f.right());
            fake::failing.clear();
            CHECK(hipGetLastError() == hipSuccess);
            CHECK(st.run == st.queued && fake::pinned.empty());
        }
}

// A stream of another device than the thread's current one: the events and the
// staging memory are the stream's device's, the current device stays.
void other_device()
{
    for (size_t n : kSizes) {
        Fields f(n), g(n);
        fake::Stream far, near;
        far.device = 1;
        CHECK(download(f.c, 2, &far) == EHD_OK && f.right());
        CHECK(fake::current == 0);
        CHECK(download(g.c, 2, &near) == EHD_OK && g.right());
    }
}

// Readers in turn on several devices keep a staging buffer each; with more of
// them than are kept the pinned memory stays bounded.
void kept(int devices)
{
    staging_retain();
    for (int round = 0; round < 5; ++round)
        for (int d = 0; d < devices; ++d) {
            Fields f(400);
            fake::Stream st;
            st.device = d;
            CHECK(download(f.c, 2, &st) == EHD_OK && f.right());
            CHECK(fake::pinned.size() <= 8);
        }
    if (devices <= 8) CHECK(fake::calls["hipHostMalloc"] == devices);
    staging_release();
}

// A read waits for the stream it was queued on, so that the runtime has done
// with its commands: left to it, they were on the bill of the box's close.
void waited()
{
    for (size_t n : kSizes) {
        Fields f(n);
        fake::Stream st;
        CHECK(download(f.c, 2, &st) == EHD_OK && f.right());
        CHECK(st.waited == st.queued);
    }
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "exact") exact();
    else if (what == "failing") failing(argv[2]);
    else if (what == "no_memory") no_memory();
    else if (what == "no_staging") no_staging(argv[2]);
    else if (what == "other_device") other_device();
    else if (what == "kept") kept(std::atoi(argv[2]));
    else if (what == "waited") waited();
    else CHECK(!"scenario");
    CHECK(fake::pinned.empty());
    std::puts("ok");
    return 0;
}
