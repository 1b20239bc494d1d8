// Elementwise kernels of the THC route.
#include "device_common.h"
#include "internal.h"

#define LAUNCH_CHECK(ctx)                                                                      \
    do {                                                                                       \
        hipError_t _e = hipGetLastError();                                                     \
        if (_e != hipSuccess)                                                                  \
            return brpa_fail((ctx), BRPA_ERR_HIP, "kernel launch failed: %s (%s:%d)",          \
                             hipGetErrorString(_e), __FILE__, __LINE__);                       \
    } while (0)

namespace {

__global__ void k_axpy(double *__restrict__ y, const double *__restrict__ x, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) y[e] += x[e];
}

}  // namespace

int launch_axpy(brpa_ctx *ctx, double *y, const double *x, int64_t n) {
    if (n <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_axpy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, y, x,
                       n);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}
