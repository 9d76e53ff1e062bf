// Functions of gw_math.h on the device, one value per thread, for the tests.
#include "gw_math.h"

namespace {

__global__ void k_quot_plain(const double *a, const double *b, double *q, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) q[i] = gw::quot_plain(a[i], b[i]);
}

}  // namespace

// q[i] = quot_plain(a[i], b[i]), host arrays; a hipError_t.
extern "C" int gw_probe_quot_plain(const double *a, const double *b, double *q, int64_t n)
{
    double *d = nullptr;
    if (n <= 0 || n > (int64_t(1) << 28)) return hipErrorInvalidValue;
    const size_t bytes = static_cast<size_t>(n) * sizeof(double);
    hipError_t e = hipMalloc(&d, 3 * bytes);
    if (e != hipSuccess) return e;
    if ((e = hipMemcpy(d, a, bytes, hipMemcpyHostToDevice)) == hipSuccess &&
        (e = hipMemcpy(d + n, b, bytes, hipMemcpyHostToDevice)) == hipSuccess) {
        hipLaunchKernelGGL(k_quot_plain, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, 0, d, d + n, d + 2 * n, n);
        if ((e = hipGetLastError()) == hipSuccess) e = hipMemcpy(q, d + 2 * n, bytes, hipMemcpyDeviceToHost);
    }
    (void)hipFree(d);
    return e;
}
