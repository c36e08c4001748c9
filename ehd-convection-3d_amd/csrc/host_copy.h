// host_copy.h -- copies from device buffers to the caller's pageable arrays
// through pinned staging memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace ehd {

// One array of a download: n elements of dev to host.
struct HostCopy {
    enum Kind {
        kFloat,          // float -> float
        kDouble,         // double -> double
        kWiden,          // float -> double
        kWidenAddMean,   // float -> double, + mean[i / plane] (mean on the device, nmean <= kMaxMean)
    };
    Kind kind;
    void* host;
    const void* dev;
    size_t n;
    const double* mean = nullptr;
    size_t nmean = 0, plane = 0;
};
constexpr size_t kMaxMean = 4096;

// Returns once the copies are complete, behind the work queued on st.
// count <= 16 arrays, at most one of them with a mean.
int download(const HostCopy* c, int count, hipStream_t st);

// The staging buffers are kept from call to call (at most eight of them) while
// any box or network is alive: the owners count themselves in and out.
void staging_retain();
void staging_release();

}  // namespace ehd
