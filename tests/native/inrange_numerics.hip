// The in-range evaluations of phx_numerics.hpp beside the plain ones, for the host (one element at a
// time, so every element takes its own path) and for the device (by waves), compared bit for bit by
// tests/test_inrange_numerics.py.  Test infrastructure only; built in-tree by __graft_entry__.build()
// (tests/native/libinrange_numerics.so).
#include <hip/hip_runtime.h>

#include "../../pyhype_amd/csrc/phx_numerics.hpp"

namespace {

// what: 0 n / d (2 values in), 1 1 / d (1), 2 limiter of a cell (7: u, dmax, dmin, hE, hW, hN, hS), 3 norm (4)
constexpr int WIDTH[4] = {2, 1, 7, 4};

__host__ __device__ inline void both(int what, const double* x, double& fast, double& plain) {
    if (what == 0) {
        fast = phx::Recip(x[1]).div(x[0]);
        plain = x[0] / x[1];
    } else if (what == 1) {
        fast = phx::Recip(x[0]).inv();
        plain = 1.0 / x[0];
    } else if (what == 2) {
        const double u = x[0], h[4] = {x[3], x[4], x[5], x[6]};
        fast = phx::limit_venkat(u, x[1], x[2], h, false);
        double p[4];
        for (int f = 0; f < 4; ++f) p[f] = phx::limit_face<false>(x[1], x[2], (u + h[f]) - u, 0);
        plain = phx::np_minimum(phx::np_minimum(phx::np_minimum(p[0], p[1]), p[2]), p[3]);
        plain = plain < 0.0 ? 0.0 : plain;
    } else {
        fast = phx::nrm4(x[0], x[1], x[2], x[3]);
        plain = phx::nrm4_ext(x[0], x[1], x[2], x[3]);
    }
}

__global__ void k_both(int what, int width, const double* in, double* fast, double* plain, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) both(what, in + (long)width * i, fast[i], plain[i]);
}

}  // namespace

extern "C" {
void inr_host(int what, const double* in, double* fast, double* plain, int n) {
    for (int i = 0; i < n; ++i) both(what, in + (long)WIDTH[what] * i, fast[i], plain[i]);
}
// device arrays; 0 on success, else the HIP error code
int inr_device(int what, const double* in, double* fast, double* plain, int n, void* stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_both, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, what, WIDTH[what], in, fast,
                       plain, n);
    return (int)hipGetLastError();
}
}
