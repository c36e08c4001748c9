// batch_harness.cpp -- drives batch.cpp on the stand-in runtime beside this
// file, the boxes and their kernels replaced by counters; tests/test_host_copy.py
// builds it and runs it with the version of the runtime that is there.
// Prints the graphs captured and replayed and the steps launched by a call of
// ehd_batch_step.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "../../ehd-convection-3d_amd/csrc/box.h"

using namespace ehd;

static long g_lbm = 0;

namespace ehd {
PopBufs pop_bufs(ehd_box*) { return {}; }
MacroBufs macro_bufs(ehd_box*) { return {}; }
bool lbm_streams(Prec, int, size_t) { return false; }
size_t lbm_f32s_batch_item_size() { return 8; }
void lbm_f32s_batch_item(void*, const LbmParams&, const PopBufs&, const MacroBufs&, unsigned, const double*) {}
hipError_t launch_lbm_f32s_batch(const void*, int, unsigned, unsigned, unsigned, bool, bool, bool, bool, hipStream_t, bool)
{
    ++g_lbm;
    return hipSuccess;
}
hipError_t launch_lbm_f64(const LbmParams&, const PopBufs&, const MacroBufs&, bool, bool, bool, bool, hipStream_t)
{
    return hipErrorInvalidValue;
}
hipError_t launch_poisson_group(Prec, const PoissonGroup&, hipStream_t) { return hipSuccess; }
PoissonShape poisson_shape(Prec, int, int, int) { return {4, 4, 16}; }
bool poisson_planes(Prec, int, int) { return false; }
}  // namespace ehd

extern "C" {
int ehd_create(const ehd_params* p, ehd_box** out)
{
    ehd_box* b = new ehd_box();
    b->prm = *p;
    b->prec = Prec::F32S;
    b->nx = p->nx;
    b->ny = p->ny;
    b->nz = p->nz;
    b->S = (size_t)p->nx * p->ny * p->nz;
    b->lp.px = p->nx;
    b->lp.SP = (unsigned)b->S;
    b->st = new fake::Stream;
    *out = b;
    return EHD_OK;
}
void ehd_destroy(ehd_box* b)
{
    delete b->st;
    delete b;
}
int ehd_init(ehd_box* b, const double*)
{
    b->initialised = true;
    return EHD_OK;
}
int ehd_diagnostics(ehd_box*, ehd_diag*) { return EHD_OK; }
}

int main(int argc, char** argv)
{
    if (argc != 3) return 2;
    fake::version = std::atoi(argv[1]);
    ehd_params p[2] = {};
    for (int i = 0; i < 2; ++i) {
        p[i].nx = p[i].ny = 32 << i;
        p[i].nz = 16;
        p[i].precision = EHD_FP32S;
    }
    ehd_batch* bt = nullptr;
    if (ehd_batch_create(p, 2, std::atoi(argv[2]), &bt) != EHD_OK || ehd_batch_init(bt, nullptr) != EHD_OK) return 3;
    const long lbm0 = g_lbm, replays0 = fake::calls["hipGraphLaunch"];
    if (ehd_batch_step(bt, 11) != EHD_OK || ehd_batch_box(bt, 0)->step != 11) return 4;
    std::printf("%ld captures, %ld replays, %ld launches\n", fake::calls["hipStreamBeginCapture"],
                fake::calls["hipGraphLaunch"] - replays0, g_lbm - lbm0);
    ehd_batch_destroy(bt);
    return 0;
}
