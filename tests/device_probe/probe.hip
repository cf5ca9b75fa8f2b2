// Device functions of the plugin that no entry point exposes by themselves, run over arrays for the GPU
// tests (test_sqrt_device_gpu.py).
#include "pt_common.h"

namespace {

__global__ void k_sqrt_1m(const float *a, float *out, float *plain, int n) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    out[i] = pgpu::sqrt_1m(a[i]);
    plain[i] = pgpu::safe_sqrt(1 - a[i]);
}

}  // namespace

// out[i] = sqrt_1m(a[i]) and plain[i] = safe_sqrt(1 - a[i]) for host arrays of n floats. Returns 0 on success.
extern "C" __attribute__((visibility("default"))) int probe_sqrt_1m(const float *a, float *out, float *plain, int n) {
    if (n <= 0 || !a || !out || !plain) return 1;
    float *d[3] = {nullptr, nullptr, nullptr};
    const size_t bytes = size_t(n) * sizeof(float);
    bool ok = true;
    for (float *&p : d) ok = ok && hipMalloc(&p, bytes) == hipSuccess;
    ok = ok && hipMemcpy(d[0], a, bytes, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(k_sqrt_1m, dim3((n + 255) / 256), dim3(256), 0, nullptr, d[0], d[1], d[2], n);
        ok = hipGetLastError() == hipSuccess;
    }
    ok = ok && hipMemcpy(out, d[1], bytes, hipMemcpyDeviceToHost) == hipSuccess &&
         hipMemcpy(plain, d[2], bytes, hipMemcpyDeviceToHost) == hipSuccess;
    for (float *p : d)
        if (p) (void)hipFree(p);
    return ok ? 0 : 1;
}
