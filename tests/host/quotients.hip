// The library's FP64 quotients on arrays, for tests/test_gpu_quotients.py:
// out[i] = qdiv(a[i], b[i]), out[n + i] = qdiv0(a[i], b[i]).
#include <hip/hip_runtime.h>

#include "tj_device.h"

__global__ void k_quotients(const double* a, const double* b, double* out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = tj::qdiv(a[i], b[i]);
    out[(size_t)n + i] = tj::qdiv0(a[i], b[i]);
}

// a, b: n device doubles; out: 2 n.  Waits for the launch; returns its status.
extern "C" int quotients(const double* a, const double* b, double* out, int n) {
    if (n < 1 || n > (1 << 24)) return -1;
    hipLaunchKernelGGL(k_quotients, dim3((n + 255) / 256), dim3(256), 0, nullptr, a, b, out, n);
    const hipError_t e = hipGetLastError();
    return (int)(e != hipSuccess ? e : hipDeviceSynchronize());
}
