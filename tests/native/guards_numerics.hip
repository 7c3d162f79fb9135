// The functions of phx_numerics.hpp that take a short evaluation where their operands are in range, beside
// the plain evaluation, for the host and for the device; compared bit for bit by
// tests/test_range_guards.py.  Test infrastructure only; built in-tree by __graft_entry__.build()
// (tests/native/libguards_numerics.so).
#include <hip/hip_runtime.h>

#include "../../pyhype_amd/csrc/phx_numerics.hpp"

namespace {

enum { DIV = 0, VENKAT, DIV_ALL, INV_AREA, PRIM2, ROE_AVG, HLLL_AVG, LIMIT_BJ, LIMIT_ODD, KINDS };
constexpr int IN[KINDS] = {2, 1, 5, 1, 8, 10, 10, 7, 7}, OUT[KINDS] = {1, 1, 4, 1, 8, 9, 8, 1, 1};

__host__ __device__ inline phx::Phys gas(double gamma, bool odd) {
    phx::Phys ph{};
    ph.gamma = gamma;
    ph.gm1 = gamma - 1.0;
    ph.one_over_gm1 = 1.0 / (gamma - 1.0);
    ph.g_over_gm1 = gamma / (gamma - 1.0);
    ph.odd_gas = odd ? 1 : 0;
    return ph;
}
__host__ __device__ inline void put(const phx::RoeAvgT<double>& m, bool hlll, double* o) {
    const double a[9] = {m.r, m.u, m.p, m.aL, m.aR, m.a, hlll ? m.eL : m.h, hlll ? m.eR : m.ia, hlll ? 0.0 : m.v};
    for (int i = 0; i < (hlll ? 8 : 9); ++i) o[i] = a[i];
}
template <bool HLLL>
__host__ __device__ inline void average(const double* x, double* fast, double* plain) {
    // x[8] = gamma, x[9] != 0: a gas that the plan marks as out of range
    const phx::Prim L{x[0], x[1], x[2], x[3]}, R{x[4], x[5], x[6], x[7]};
    const phx::Phys ph = gas(x[8], x[9] != 0.0);
    put(phx::roe_avg<HLLL>(L, R, ph), HLLL, fast);
    phx::RoeAvgT<double> m;
    phx::roe_avg_f<false, HLLL>(L, R, ph, m);
    put(m, HLLL, plain);
}
// limiter value of a cell from the four faces' values in the reference's order
template <bool GEN>
__host__ __device__ inline double four_faces(const double* x, int lim) {
    double p[4];
    for (int f = 0; f < 4; ++f) p[f] = phx::limit_face<GEN>(x[1], x[2], (x[0] + x[3 + f]) - x[0], lim);
    const double m = phx::np_minimum(phx::np_minimum(phx::np_minimum(p[0], p[1]), p[2]), p[3]);
    return m < 0.0 ? 0.0 : m;
}

__host__ __device__ inline void both(int what, const double* x, double* fast, double* plain) {
    const double h[4] = {x[3], x[4], x[5], x[6]};
    switch (what) {
        case DIV: fast[0] = phx::Recip(x[1]).div(x[0]); plain[0] = x[0] / x[1]; break;
        case VENKAT: fast[0] = phx::venkat_in_range(x[0]); plain[0] = phx::venkatakrishnan_fn(x[0]); break;
        case DIV_ALL: {
            const double n[4] = {x[0], x[1], x[2], x[3]};
            double q[4];
            phx::div_all(n, x[4], q);
            for (int i = 0; i < 4; ++i) { fast[i] = q[i]; plain[i] = n[i] / x[4]; }
            break;
        }
        case INV_AREA: fast[0] = phx::inv_area(x[0]); plain[0] = 1.0 / x[0]; break;
        case PRIM2: {
            const phx::Q4 a{{x[0], x[1], x[2], x[3]}}, b{{x[4], x[5], x[6], x[7]}};
            const phx::Phys ph = gas(1.4, false);
            phx::Prim L, R;
            phx::cons_to_prim2(a, b, ph, L, R);
            const phx::Prim l = phx::cons_to_prim(a, ph), r = phx::cons_to_prim(b, ph);
            const double f[8] = {L.r, L.u, L.v, L.p, R.r, R.u, R.v, R.p}, g[8] = {l.r, l.u, l.v, l.p, r.r, r.u, r.v, r.p};
            for (int i = 0; i < 8; ++i) { fast[i] = f[i]; plain[i] = g[i]; }
            break;
        }
        case ROE_AVG: average<false>(x, fast, plain); break;
        case HLLL_AVG: average<true>(x, fast, plain); break;
        case LIMIT_BJ: fast[0] = phx::limit_bj(x[0], x[1], x[2], h); plain[0] = four_faces<true>(x, 1); break;
        default: fast[0] = phx::limit_venkat(x[0], x[1], x[2], h, true); plain[0] = four_faces<false>(x, 0); break;
    }
}

constexpr int MAX_IN = 10, MAX_OUT = 9;

__host__ __device__ inline void element(int what, const double* in, double* fast, double* plain, long i, int nin, int nout) {
    double x[MAX_IN], f[MAX_OUT], p[MAX_OUT];
    for (int k = 0; k < MAX_IN; ++k) x[k] = k < nin ? in[i * nin + k] : 0.0;
    both(what, x, f, p);
    for (int k = 0; k < nout; ++k) { fast[i * nout + k] = f[k]; plain[i * nout + k] = p[k]; }
}

__global__ void k_guards(int what, int nin, int nout, const double* in, double* fast, double* plain, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) element(what, in, fast, plain, i, nin, nout);
}

}  // namespace

extern "C" {
int rg_in(int what) { return IN[what]; }
int rg_out(int what) { return OUT[what]; }
void rg_host(int what, const double* in, double* fast, double* plain, int n) {
    for (int i = 0; i < n; ++i) element(what, in, fast, plain, i, IN[what], OUT[what]);
}
// device arrays; 0 on success, else the HIP error code
int rg_device(int what, const double* in, double* fast, double* plain, int n, void* stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_guards, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, what, IN[what], OUT[what], in,
                       fast, plain, n);
    return (int)hipGetLastError();
}
}
