// march_device.hip - the kernels' reciprocal, quotient and square root
// (lum_amd/csrc/march.hpp, the GPU's branch) over arrays, for
// tests/test_gpu_arithmetic.py.  Compiled by __graft_entry__.build().
#include "../lum_amd/csrc/march.hpp"

using namespace lumx;

namespace {
__global__ __launch_bounds__(256) void apply_kernel(int op, const float* a, const float* d, float* out, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float y = d[i];
    out[i] = op == 0 ? rcp_rn(y) : op == 1 ? div_rn(a[i], y, rcp_rn(y)) : sqrt_rn(y);
}
}  // namespace

// out[i] = 1 / d[i] (op 0), a[i] / d[i] (1), sqrt(d[i]) (2), device arrays of
// n elements; returns when they are written.
extern "C" int md_apply(int op, const float* a, const float* d, float* out, int n) {
    if (n <= 0 || !d || !out || (op == 1 && !a)) return -1;
    hipLaunchKernelGGL(apply_kernel, dim3((n + 255) / 256), dim3(256), 0, nullptr, op, a, d, out, n);
    if (hipGetLastError() != hipSuccess) return -2;
    return hipDeviceSynchronize() == hipSuccess ? 0 : -3;
}
