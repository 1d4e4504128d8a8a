// fill.hip -- multi-region fill kernel and the library's error bookkeeping.
#include <cstdarg>

#include "fill.h"

namespace sessd {

namespace {
thread_local char g_last_error[1024] = "";  // (reporting that memory has run out takes none)
}

int fail(int code, const char* fmt, ...) {
    char buf[sizeof(g_last_error)];  // (an argument may be the last message)
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    std::memcpy(g_last_error, buf, sizeof(buf));
    return code;
}

const char* last_error_cstr() { return g_last_error; }

template <int N>
__global__ void __launch_bounds__(256) fill_kernel(FillPlan<N> p) {
    fill_pass(p, blockIdx.x);
}

template <int N>
static int launch_fill_n(const FillArgs& a, hipStream_t stream) {
    FillPlan<N> p;
    const int blocks = make_fill_plan(a, p);
    if (blocks < 0) return fail(SESSD_E_INVALID, "fill: a region is not 16-byte aligned");
    hipLaunchKernelGGL(fill_kernel<N>, dim3(blocks), dim3(256), 0, stream, p);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

int launch_fill(const FillArgs& a, hipStream_t stream) {
    if (a.n == 0) return SESSD_OK;
    return a.n <= kFewRegions ? launch_fill_n<kFewRegions>(a, stream) : launch_fill_n<FillArgs::kMaxRegions>(a, stream);
}

}  // namespace sessd
