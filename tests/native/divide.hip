// Division as the kernels do it (DivBy) and as the compiler does it, for a test:
// n numerators a over denominators b, and a / 3 with the reciprocal given.
// Host pointers; returns the first HIP error.
#include <hip/hip_runtime.h>

#include "fv3d_device.h"

using namespace fv3d;

__global__ void k_divide(long n, const double *a, const double *b, double *out)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    out[t] = DivBy(b[t]).of(a[t]);
    out[n + t] = a[t] / b[t];
    out[2 * n + t] = DivBy(3.0, 1.0 / 3.0).of(a[t]);
    out[3 * n + t] = a[t] / 3.0;
}

extern "C" int test_divide(long n, const double *a, const double *b, double *out)
{
    double *d = nullptr;
    hipError_t e = hipMalloc(&d, 6 * n * sizeof(double));
    if (e != hipSuccess) return e;
    e = hipMemcpy(d, a, n * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d + n, b, n * sizeof(double), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_divide, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, n, d, d + n, d + 2 * n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d + 2 * n, 4 * n * sizeof(double), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return e;
}
