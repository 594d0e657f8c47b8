// One FP64 form of tp_fp64.h per call, evaluated on the device: the branches the kernels take (hardware reciprocal,
// exponent and mantissa from the high word, the device's table), which a host build does not contain.
#include "tp_fp64.h"

__global__ void k_form(int what, int n, const double *x, double *y)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = x[i];
    double r = 0;
    switch (what) {
    case 0: r = tp_fp64_exp(v); break;
    case 1: r = tp_fp64_log(v); break;
    case 2: r = tp_fp64_rcp(v); break;
    case 3: r = tp_fp64_log1p(v); break;
    case 4: r = tp_fp64_exp10(v); break;
    case 5: r = tp_fp64_exp_any(v); break;
    case 6: r = tp_fp64_exp_low(v); break;
    case 7: r = tp_fp64_rcp_any(v); break;
    }
    y[i] = r;
}

extern "C" int run(int what, int n, const double *x, double *y)
{
    if (n <= 0 || n > 1 << 24 || what < 0 || what > 7) return 1;
    double *d = nullptr;
    const size_t b = (size_t)n * sizeof(double);
    if (hipMalloc(&d, 2 * b) != hipSuccess) return 2;
    bool ok = hipMemcpy(d, x, b, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(k_form, dim3((n + 255) / 256), dim3(256), 0, 0, what, n, d, d + n);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(y, d + n, b, hipMemcpyDeviceToHost) == hipSuccess;
    }
    return hipFree(d) == hipSuccess && ok ? 0 : 3;
}
