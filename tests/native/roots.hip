// The square root and the quotient of the pair sums over given arguments, for
// tests/test_gpu_roots.py.
#include "sphg_roots.h"

namespace {

__global__ void k_roots(const double* a, const double* b, double* root, double* quotient, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    root[i] = sphg::sqrt_n(a[i]);
    quotient[i] = sphg::div_n(a[i], b[i]);
}

}  // namespace

// out: n roots of a, then n quotients a / b; the HIP error, 0 for none
extern "C" int roots(const double* a, const double* b, double* out, int n) {
    if (n <= 0) return 0;
    const size_t bytes = sizeof(double) * (size_t)n;
    double* d = nullptr;
    hipError_t e = hipMalloc(&d, 4 * bytes);
    if (e != hipSuccess) return (int)e;
    e = hipMemcpy(d, a, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d + n, b, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_roots, dim3((n + 255) / 256), dim3(256), 0, nullptr, d, d + n, d + 2 * (size_t)n,
                           d + 3 * (size_t)n, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d + 2 * (size_t)n, 2 * bytes, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return (int)e;
}
