// phx_stage.hpp -- gfx950 stage kernels of the pyHype MUSCL/RK backend.
//
// Stage kernel design ("rolling rows"): one wavefront owns a strip of 60 columns of one block
// plus two halo lanes on each side and walks up a range of rows.  Per row it loads one row of the
// stage state, reconstructs each cell once (Green-Gauss + Venkatakrishnan + limited face states),
// evaluates each x-face flux once (lane j computes face j-1|j and hands it to lane j-1 through a
// cross-lane shuffle), evaluates the y-face between this row and the previous one in registers
// (same lane), finishes the residual of the previous row and applies every Butcher update of the
// stage in the same pass.  Ghost cells (inter-block neighbours, reflected walls, outlets) are
// produced on the fly from the stage state, so there is no separate ghost-fill pass.  The last
// stage of a step also reduces the CFL time step of the next step and the realizability flag.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "../../include/pyhype_hip.h"
#include "phx_adjoint_ops.hpp"
#include "phx_device.hpp"
#include "phx_numerics.hpp"
#include "phx_plan.hpp"

namespace phx {
namespace stage {

using namespace phx::dev;
using namespace phx::host;

constexpr int WAVE = 64;
constexpr int HALO = 2;
constexpr int STRIP = WAVE - 2 * HALO;  // owned columns per wavefront
constexpr unsigned long long DT_INF_BITS = 0x7FF0000000000000ull;  // +inf
// The CFL minimum of a case is accumulated in nslot partial minima (a power of two, at most
// DT_SLOTS), each on a cache line of its own (DT_STRIDE words apart): the waves of a stage spread
// their atomicMin over the slots instead of serialising on one address, and step_dt or k_finalize takes
// the minimum over the slots (an exact operation, independent of the order).  Plans with many cases
// use fewer slots per case (their waves are spread over the cases already).
constexpr int DT_SLOTS = 64;
constexpr int DT_STRIDE = 16;
__host__ __device__ constexpr long dt_slot(int c, int slot, int nslot) { return ((long)c * nslot + slot) * DT_STRIDE; }
__device__ __forceinline__ int wave_slot(int nslot) {
    return (int)((blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE) & (nslot - 1));
}

// A work item as the kernels read it: with the descriptor of its block, so that the first values a
// wave computes addresses from arrive after one scalar load instead of two in a row (about 0.2 us of
// every launch, more where the descriptors are not in the cache yet).
struct DevItem {
    int block, j0, r0, r1;
    DevBlock b;
};

// Every per-item function below is __forceinline__, so that no kernel makes a device-function call.
// Outlined (s_swappc) item functions of the HLLL Gauss-face and generic shared-halo kernels, which
// appeared when the HLLL norm grew, returned NaN residuals on gfx950 (ROCm 7.2) where the same
// source inlined, and a stand-alone kernel of the same flux, are bit-exact.

// Closing one step and opening the next: the time steps from the CFL minima of the state (or a given
// schedule), the times and the step counter.  As a kernel of its own between two steps this took 2.7 to
// 4.6 us and a launch gap; the stage kernels take it along in extra workgroups instead, where nothing
// waits for it:
//  * FOLD_ALL: the first kernel of a step's first stage that only reconstructs, into scratch (split and
//    element-wise stages); the step's later kernels read dt.
//  * FOLD_DT, FOLD_TIME: the shared-halo stage needs dt in the step's only kernel per stage, so in the
//    first stage every update wave takes the minimum itself while extra workgroups store dt and the
//    counter, and in the second, when nobody reads them any more, the times and the cleared minima.
// The minima are kept in two sets, read and written by turns, since a two-stage step writes the next
// step's minima in the launch that clears this step's.
enum { FOLD_NONE = 0, FOLD_ALL, FOLD_DT, FOLD_TIME };
constexpr int NEVER = 0x7fffffff;  // bad[] of a case that never failed
struct StepFold {  // in device memory, read where it is used: as kernel arguments it costs every wave registers
    int ncases;
    double cfl;
    unsigned long long* dtmin;
    const double* tfinal;
    double* t;
    double* dt;
    int* step;
};

struct StageArgs {
    const DevBlock* blocks;
    const DevItem* items;
    int nitems;
    int nout;
    int state_out;
    const double* Uin;
    const double* dt;
    double* Rout;
    double* dst[MAX_OUT];
    const double* src[MAX_OUT];
    double a[MAX_OUT];
    unsigned long long* dtmin;
    int* bad;          // per case: first step whose result was unrealizable (INT_MAX = none)
    const int* step;   // index of the step being computed (1-based)
    int skip_dead;     // skip the blocks of cases that failed at an earlier step
    int rows_wave;     // shared-halo and y-face stages: rows per workgroup
    double* sn;        // split stage: limited N and S states per cell (8 doubles, offset 2*off)
    double* p1;        // split stage: LW*(2 FW) - LE*(2 FE) per cell (4 doubles, state layout)
    double* yf;        // split stage: y-face fluxes (DevBlock::yoff)
    double* rb;        // element-wise stage: limited face states E, W, N, S per cell (16 doubles)
    double* ff;        // element-wise stage: face fluxes (4 doubles per face, DevBlock::foff)
    int nslot;         // partial CFL minima per case
    int fq;            // flat y-face stage: LDS faces per lane
    int fold_mode;     // what the launch takes along (FOLD_*), for the minima's set fold_set
    int fold_set;
    int fold_blocks;   // extra workgroups of this launch, behind the others
    const StepFold* fold;
    const double* frozen;  // the schedule's time steps instead of the CFL minima
    Phys ph;
};

// Element i of an array that no kernel writes, as a reference through the constant address
// space: uniform field reads become scalar loads that the compiler may repeat instead of keeping
// the whole element in registers.
template <class T>
__device__ __forceinline__ const T& const_ref(const T* p, long i) {
    return *(const T*)(((const __attribute__((address_space(4))) T*)p) + i);
}

// Whether the block's case became unrealizable at an earlier step: it is frozen, as the reference aborts
// that run (Euler2D.py:144-152).  Scalar loads (a lane that fails in this stage writes the current step,
// which leaves the comparison as it is); a kernel asks after it has issued its first loads, which do
// not wait for the answer then.  In a launch whose extra workgroups advance the counter the answer does not
// depend on it where states are written (FOLD_DT: every failure on record is an earlier step's); a
// FOLD_ALL launch writes scratch only, which the step's next kernel does not use for a frozen case.
__device__ __forceinline__ bool frozen_case(const StageArgs& A, const DevBlock& B) {
    return A.skip_dead && ld_const(A.bad, B.case_id) < (A.fold_mode == FOLD_DT ? NEVER : ld_const(A.step, 0));
}

// dt of case c, which an aligned group of nslot lanes asks for together: CFL * minimum, clipped to
// t_final - t (solvers/base.py:126-136)
__device__ __forceinline__ double step_dt(const StageArgs& A, int c) {
    if (A.frozen != nullptr) return A.frozen[c];
    const StepFold& F = const_ref(A.fold, 0);
    unsigned long long m = F.dtmin[dt_slot(A.fold_set * F.ncases + c, threadIdx.x & (A.nslot - 1), A.nslot)];
    const double rem = F.tfinal[c] - F.t[c];
    for (int o = A.nslot / 2; o > 0; o >>= 1) {
        const unsigned long long x = __shfl_xor(m, o, A.nslot);
        m = x < m ? x : m;
    }
    const double d = F.cfl * __longlong_as_double((long long)m);
    return rem < d ? rem : d;
}

// The extra workgroups of a launch (their first wave; nslot lanes per case); false in the others.
__device__ __forceinline__ bool fold_step(const StageArgs& A) {
    const int e = (int)blockIdx.x - ((int)gridDim.x - A.fold_blocks);
    if (e < 0) return false;
    const StepFold& F = const_ref(A.fold, 0);
    if (threadIdx.x >= WAVE) return true;
    const int c = e * (WAVE / A.nslot) + (int)threadIdx.x / A.nslot;
    const int g = threadIdx.x & (A.nslot - 1);
    if (c < F.ncases) {
        if (A.fold_mode == FOLD_TIME) {
            if (g == 0) F.t[c] += F.dt[c];
        } else {
            double d = step_dt(A, c);
            if (A.bad[c] != NEVER) d = 0.0;  // a failed case keeps its time
            if (g == 0) {
                F.dt[c] = d;
                if (A.fold_mode == FOLD_ALL) F.t[c] += d;  // Euler2D.py:209
            }
        }
        if (A.fold_mode != FOLD_DT) F.dtmin[dt_slot(A.fold_set * F.ncases + c, g, A.nslot)] = DT_INF_BITS;
    }
    if (A.fold_mode != FOLD_TIME && e == 0 && threadIdx.x == 0) F.step[0] += 1;
    return true;
}

// Cross-lane moves of a 4-vector by one lane (the end lanes keep their value), in two forms: through the
// LDS pipe (ds_bpermute_b32), and as v_mov_b32 with a wave shift, two to a double.  The first leaves the
// vector pipe to the arithmetic that bounds the fused stage (batch of 2.4 x 10^6 cells, 8 steps: 6,423
// us, with shifts 6,772); the second has no latency for a wave to wait out, which is what the split
// stage's reconstruction does (5 x 500^2 HLLL, 16 steps: 3,128 us, with shifts 3,059).
__device__ __forceinline__ Q4 shfl_up1(const Q4& q) {
    Q4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r.v[k] = __shfl_up(q.v[k], 1, WAVE);
    return r;
}
__device__ __forceinline__ Q4 shfl_down1(const Q4& q) {
    Q4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r.v[k] = __shfl_down(q.v[k], 1, WAVE);
    return r;
}
template <int CTRL>
__device__ __forceinline__ Q4 wave_shift(const Q4& q) {
    Q4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, q.v[k]);
        const int lo = (int)(unsigned)b, hi = (int)(unsigned)(b >> 32);
        const unsigned l = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
        const unsigned h = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
        r.v[k] = __builtin_bit_cast(double, ((unsigned long long)h << 32) | l);
    }
    return r;
}
__device__ __forceinline__ Q4 shift_up1(const Q4& q) { return wave_shift<0x138>(q); }    // wave_shr:1
__device__ __forceinline__ Q4 shift_down1(const Q4& q) { return wave_shift<0x130>(q); }  // wave_shl:1

// Outputs of the stage program are written in chunks of EMIT_CHUNK: the chunk's sources are loaded
// together before its stores (an output's source is never a buffer an earlier output of the stage
// writes), and the chunk loop is not unrolled, so the outputs' pointers and coefficients are read
// from the kernel arguments per chunk instead of occupying scalar registers for all MAX_OUT slots.
constexpr int EMIT_CHUNK = 3;

// Sources of the first output chunk of owned cell (kk, j), loaded ahead of the row's arithmetic so
// that their latency overlaps it.  Only this lane writes these cells in this stage (after it has
// read them), so the early read returns what emit_row would read.
__device__ __forceinline__ void prefetch_sources(const StageArgs& A, const DevBlock& B, int kk, int j,
                                                 Q4 (&pre)[EMIT_CHUNK]) {
    const long idx = B.off + 4 * ((long)kk * B.nx + j);
#pragma unroll
    for (int q = 0; q < EMIT_CHUNK; ++q)
        if (q < A.nout) pre[q] = ld4(A.src[q] + idx);
}

// Residual of owned cell (kk, j) -> every Butcher output of the stage program
// (explicit_runge_kutta.py:63-80); on the last stage also the cell's CFL quantity and realizability.
// PF: the first chunk's sources were loaded by prefetch_sources into pre; on a Cartesian block dxc
// is the cell's column width and the row height a scalar load.
template <bool CART, bool PF = false>
__device__ __forceinline__ void emit_row(const StageArgs& A, const DevBlock& B, int kk, int j, double dt, const Q4& Res,
                                         double& lane_dt, bool& lane_bad, const Q4* pre = nullptr,
                                         double dxc = 0.0) {
    const long idx = B.off + 4 * ((long)kk * B.nx + j);
    if (A.Rout) st4(A.Rout + idx, Res);
#pragma unroll 1
    for (int m0 = 0; m0 < A.nout; m0 += EMIT_CHUNK) {
        Q4 s[EMIT_CHUNK];
        if (PF && m0 == 0) {
#pragma unroll
            for (int q = 0; q < EMIT_CHUNK; ++q) s[q] = pre[q];
        } else {
#pragma unroll
            for (int q = 0; q < EMIT_CHUNK; ++q)
                if (m0 + q < A.nout) s[q] = ld4(A.src[m0 + q] + idx);
        }
#pragma unroll
        for (int q = 0; q < EMIT_CHUNK; ++q) {
            const int m = m0 + q;
            if (m >= A.nout) break;
            Q4 o;
            const double am = A.a[m];
            if (am == 0.0) {
                o = s[q];
            } else {
                const double cdt = dt * am;  // dt * a[stage][step] (explicit_runge_kutta.py:72)
#pragma unroll
                for (int c = 0; c < 4; ++c) o.v[c] = s[q].v[c] + cdt * Res.v[c];
            }
            st4(A.dst[m] + idx, o);
            if (m == A.state_out && A.dtmin != nullptr) {
                double dx, dy;
                if (PF && CART) {
                    dx = dxc;
                    dy = CartGT<true>{B.geom, B.nx, B.ny}.row(R_dy, kk);
                } else {
                    cell_dxdy<CART>(B, kk, j, dx, dy);
                }
                const double t = phx::cell_dt(o, dx, dy, A.ph);
                if (!(o.v[0] > 0.0) || !(o.v[3] > 0.0) || !(t == t)) lane_bad = true;
                else lane_dt = fmin(lane_dt, t);
            }
        }
    }
}

// wave-level min of the CFL quantities and any-unrealizable of one work item -> per-case atomics
__device__ __forceinline__ void reduce_item(const StageArgs& A, const DevBlock& B, int lane, double lane_dt,
                                            bool lane_bad) {
    if (A.dtmin != nullptr) {
        double m = lane_dt;
#pragma unroll
        for (int o = WAVE / 2; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o, WAVE));
        const bool anybad = __any(lane_bad);
        if (lane == 0) {
            const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
            if (bits < DT_INF_BITS) atomicMin(&A.dtmin[dt_slot(B.case_id, wave_slot(A.nslot), A.nslot)], bits);
            if (anybad) atomicMin(&A.bad[B.case_id], *A.step);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// one work item of one RK stage
// ---------------------------------------------------------------------------------------------
// PF (the instances with a budget of 2 waves per SIMD, which have registers to spare): the block
// descriptor is read through the constant address space (scalar loads), and each row iteration
// issues its loads in the order they are needed, before its arithmetic: the row's geometry and face
// lengths, then the next row's states and the sources of the row it emits.  Vector-memory waits
// are in issue order, so the wait for the geometry leaves the later loads in flight.  On Cartesian
// blocks the column arrays are loaded once per item and the cell areas one row ahead, so the only
// geometry a row iteration waits for was requested an iteration earlier.
template <bool CART, int FLUX, bool GEN, bool PF = false>
__device__ __forceinline__ void stage_item(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = PF ? it.b : A.blocks[it.block];
    // a case that became unrealizable is frozen: the reference aborts that run (Euler2D.py:144-152)
    if (frozen_case(A, B)) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int nx = B.nx, ny = B.ny;
    const int j = it.j0 - HALO + lane;
    const bool valid = (j >= -1) && (j <= nx);
    const bool inner = (j >= 0) && (j < nx);
    const bool gcol = (j == -1) || (j == nx);
    const bool recon = inner && (j >= it.j0 - 1) && (j <= it.j0 + STRIP);
    const bool xface = (j >= it.j0) && (j <= min(it.j0 + STRIP, nx));
    const bool owner = inner && (j >= it.j0) && (j < it.j0 + STRIP);
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    const Phys ph = A.ph;

    const int kr0 = max(it.r0 - 1, 0);
    const int kr1 = min(it.r1, ny);  // row ny is a virtual row closing the north boundary face

    Q4 Um = phx::q4zero(), Uc = phx::q4zero(), Up = phx::q4zero();
    if (inner) Um = fetch_r<CART, GEN>(A.blocks, B, A.Uin, kr0 - 1, j, ph);
    if (valid) Uc = fetch_r<CART, GEN>(A.blocks, B, A.Uin, kr0, j, ph);

    Q4 QNprev = phx::q4zero(), part = phx::q4zero();
    double prevLN = 0.0, prevA = 1.0;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;

    // Cartesian blocks: the column arrays once per item, the cell areas one row ahead, the row
    // arrays as scalar loads
    const CartGT<true> CG{B.geom, nx, ny};
    CartCols cols{};
    double Acur = 1.0, Anext = 1.0;
    if (PF && CART && inner) {
        cols = cart_cols<true>(B, j);
        Acur = CG.A(kr0, j);
    }

    Q4 pre[EMIT_CHUNK];
    for (int k = kr0; k <= kr1; ++k) {
        const bool real = (k < ny);
        const bool xrow = (k >= it.r0) && (k < it.r1);
        phx::CellGeo g;
        double LW = 0.0, LE = 0.0, LS = 0.0, LN = 0.0, Ac = 1.0;
        if (PF && CART) {
            if (real && recon) g = cart_cell_geo<true>(B, cols, k, Acur);
            if (xrow && owner) {
                LW = CG.row(R_LW, k); LE = CG.row(R_LE, k);
                LS = cols.LS; LN = cols.LN;
                Ac = Acur;
            }
        } else if (PF) {
            if (real && recon) g = cell_geo<CART>(B, k, j);
            if (xrow && owner) cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        }
        if (real) {
            if (inner) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
            else if (gcol && k + 1 <= kr1 && k + 1 < ny) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
        }
        if (PF && owner && k - 1 >= it.r0) prefetch_sources(A, B, k - 1, j, pre);
        if (PF && CART && inner && k + 1 < ny) Anext = CG.A(k + 1, j);
        const Q4 Uw = shfl_up1(Uc);
        const Q4 Ue = shfl_down1(Uc);
        phx::Recon r;
        r.E = r.W = r.N = r.S = phx::q4zero();
        if (real && recon) {
            if (!PF) g = cell_geo<CART>(B, k, j);
            r = phx::reconstruct<GEN>(Uc, Uw, Ue, Um, Up, g, ph.limiter);
        }
        const Q4 qsend = (j == -1) ? Uc : r.E;
        const Q4 QEl = shfl_up1(qsend);  // limited east state of cell j-1 (ghost value for j == 0)
        Q4 FW = phx::q4zero();
        if (xrow && xface) {
            const Q4 L = (j == 0) ? outer_state<CART>(B, PHX_W, r.W, QEl, k, j) : QEl;
            const Q4 R = (j == nx) ? outer_state<CART>(B, PHX_E, QEl, Uc, k, j) : r.W;
            FW = xflux<CART, FLUX, GEN>(B, L, R, k, j, ph);
        }
        const Q4 FE = shfl_down1(FW);  // flux of face j+1 (east face of cell j)

        if (k >= it.r0 && owner) {
            // face between rows k-1 and k (south face of row k, north face of row k-1)
            const Q4 L = (k == 0) ? outer_state<CART>(B, PHX_S, r.S, Um, k, j) : QNprev;
            const Q4 R = (k == ny) ? outer_state<CART>(B, PHX_N, QNprev, Uc, k - 1, j) : r.S;
            const Q4 F = yflux<CART, FLUX, GEN>(B, L, R, k, j, ph);
            if (k - 1 >= it.r0) {
                // residual of row k-1: 0.5*(W - E + S - N)/A with I = L*(2*F) (fvm/base.py:141-190)
                const int kk = k - 1;
                Q4 Res;
#pragma unroll
                for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * (part.v[c] - prevLN * (2.0 * F.v[c]));
                phx::div_all(Res.v, prevA, Res.v);
                emit_row<CART, PF>(A, B, kk, j, dt, Res, lane_dt, lane_bad, pre, cols.dx);
            }
            if (xrow) {
                if (!PF) cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    part.v[c] = (LW * (2.0 * FW.v[c]) - LE * (2.0 * FE.v[c])) + LS * (2.0 * F.v[c]);
                prevLN = LN;
                prevA = Ac;
            }
        }
        QNprev = r.N;
        Um = Uc;
        Uc = Up;
        Acur = Anext;
    }

    reduce_item(A, B, lane, lane_dt, lane_bad);
}

// Work distribution: 8 XCDs receive workgroups round-robin; each XCD gets a contiguous range of the
// (spatially ordered) work list so that halo rows/columns shared by neighbouring items are reused
// from the same L2.
__device__ __forceinline__ void item_range(int n, int& lo, int& hi, int& first, int& stride, int extra = 0) {
    const int G = (int)gridDim.x - extra, w = blockIdx.x;
    if (G >= 8) {
        const int x = w & 7;
        lo = (int)(((long)n * x) >> 3);
        hi = (int)(((long)n * (x + 1)) >> 3);
        first = lo + (w >> 3);
        stride = (G - x + 7) >> 3;
    } else {
        lo = 0; hi = n; first = w; stride = G;
    }
}

// MINW: minimum waves per SIMD the register allocation must allow (2 or 3; tuned per workload)
// GEN: limiter other than Venkatakrishnan, selected at run time
template <bool CART, int FLUX, int MINW, bool GEN>
__global__ void __launch_bounds__(WAVE, MINW) k_stage(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) stage_item<CART, FLUX, GEN, MINW == 2>(A, const_ref(A.items, i));
}

// ---------------------------------------------------------------------------------------------
// shared-halo stage: one launch per stage for small meshes, where the time of a stage is the chain of one
// wave, the latency of its loads and the instructions it runs for the first time (about 2 us of 10 went
// into fetching them).  A workgroup takes R = 1 or 2 cell rows [r0, r1) of one strip with 4 (R + 2) waves:
//   1. wave 4 i + v reconstructs variable v of row r0 - 1 + i (the outer two rows are halo) and writes
//      the limited face states to LDS (the value itself beyond a block side);
//   2. one wave per face row takes an x-face row or a y-face row from there, flux to LDS, while
//   3. one wave per cell row loads what the update needs, and completes its row after the barrier.
// A wave's chain is one variable's reconstruction, then one flux or one update, and every wave of a
// phase runs the same code (one reconstruction, one flux), a third of the instructions of a wave that does
// a whole row.  Compared with the split stage's two kernels it saves a launch (1 us between two kernels,
// 2 until the first values have arrived) and the states and fluxes that pass through memory; the
// price is (R + 2)/R of the reconstructions.  Same arithmetic and association order as stage_item.
// ---------------------------------------------------------------------------------------------
constexpr int WG_MAX_ROWS = 2;
__host__ __device__ inline int wg_rows(int rows_per_item) { return rows_per_item > 1 ? WG_MAX_ROWS : 1; }
constexpr int wg_waves(int rows) { return 4 * (rows + 2); }

// doubles of LDS: E and W states of R rows, N and S of R + 1, x-fluxes of R rows, y-fluxes of R + 1
constexpr int WG_PLANE = 4 * WAVE;
constexpr int wg_lds(int rows) { return (6 * rows + 3) * WG_PLANE; }

__device__ __forceinline__ double pick(const Q4& q, int v) {
    return v == 0 ? q.v[0] : (v == 1 ? q.v[1] : (v == 2 ? q.v[2] : q.v[3]));
}

// Variable v of the stage state at row k of a wave's strip (k and v are the same for the whole wave, so
// the row's place in the block is decided by scalar branches), in the reconstruction variables: cells at
// the `inner` columns, ghost values beyond the south and north sides and, with GC in waves at a block
// side (`edge`), at the two ghost columns.
template <bool CART, bool GEN, bool GC>
__device__ __forceinline__ double row_value(const StageArgs& A, const DevBlock& B, int k, int j, int v, bool inner,
                                            bool edge) {
    const bool inside = k >= 0 && k < B.ny;
    const bool prim = GEN && A.ph.prim;
    double x = 0.0;
    if (inside && !prim && inner) x = gld(A.Uin, B.off + 4 * ((long)k * B.nx + j) + v);
    if (!inside || prim || (GC && edge)) {
        Q4 q = phx::q4zero();
        bool full = false;
        if (!inside) {
            if (inner) q = k < 0 ? ghost_value<CART, PHX_S>(A.blocks, B, A.Uin, k, j) : ghost_value<CART, PHX_N>(A.blocks, B, A.Uin, k, j);
            full = inner;
        } else {
            if (prim && inner) {
                q = ld4(A.Uin + B.off + 4 * ((long)k * B.nx + j));
                full = true;
            }
            if (GC && edge) {
                if (j == -1) q = ghost_value<CART, PHX_W>(A.blocks, B, A.Uin, k, j);
                if (j == B.nx) q = ghost_value<CART, PHX_E>(A.blocks, B, A.Uin, k, j);
                full = full || j == -1 || j == B.nx;
            }
        }
        if (prim) q = phx::prim_q4(phx::cons_to_prim(q, A.ph));
        if (full) x = pick(q, v);
    }
    return x;
}

template <bool CART, int FLUX, int R, bool GEN>
__device__ __forceinline__ void stage_wg_item(const StageArgs& A, const DevItem& it, double* lds) {
    const DevBlock B = it.b;  // in scalar registers
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int nx = B.nx, ny = B.ny, nrow = it.r1 - it.r0;  // (the last item of a strip may be shorter)
    const int j = it.j0 - HALO + lane;
    const bool inner = (j >= 0) && (j < nx);
    const bool owner = inner && (j >= it.j0) && (j < it.j0 + STRIP);
    const bool west = it.j0 == 0, east = it.j0 + STRIP + HALO > nx;  // strips that touch the block's sides
    double* const sE = lds;                                // [R][4][WAVE]: face states of row r0 + i
    double* const sW = sE + R * WG_PLANE;
    double* const sN = sW + R * WG_PLANE;                  // [R + 1]: N states of row r0 - 1 + i
    double* const sS = sN + (R + 1) * WG_PLANE;            // [R + 1]: S states of row r0 + i
    double* const fX = sS + (R + 1) * WG_PLANE;            // [R]: x-fluxes of row r0 + i
    double* const fY = fX + R * WG_PLANE;                  // [R + 1]: y-fluxes of face row r0 + i

    {   // one variable of one row
        const int i = w >> 2, v = w & 3, k = it.r0 - 1 + i;
        const bool used = i <= nrow + 1;
        const bool real = used && k >= 0 && k < ny;
        const bool recon = real && inner && (j >= it.j0 - 1) && (j <= it.j0 + STRIP);
        double c = 0.0, m = 0.0, p = 0.0;
        phx::CellGeo g;
        if (used) c = row_value<CART, GEN, true>(A, B, k, j, v, inner, west || east);
        if (real) {
            m = row_value<CART, GEN, false>(A, B, k - 1, j, v, inner, false);
            p = row_value<CART, GEN, false>(A, B, k + 1, j, v, inner, false);
            if (recon) g = cell_geo<CART>(B, k, j);
        }
        // a frozen case leaves here (uniform over the workgroup; nothing has been written)
        if (frozen_case(A, B)) return;
        const double e = __shfl_down(c, 1, WAVE), we = __shfl_up(c, 1, WAVE);
        double qE = c, qW = c, qN = c, qS = c;
        if (recon) phx::reconstruct_var<GEN>(c, we, e, m, p, g, A.ph.limiter, qE, qW, qN, qS);
        const int at = v * WAVE + lane;
        if (i >= 1 && i <= nrow) {
            sE[(i - 1) * WG_PLANE + at] = qE;
            sW[(i - 1) * WG_PLANE + at] = qW;
        }
        if (i <= nrow) sN[i * WG_PLANE + at] = qN;
        if (i >= 1 && used) sS[(i - 1) * WG_PLANE + at] = qS;
    }
    constexpr int WAVES = wg_waves(R);
    const int u = w - (WAVES - R);  // the last R waves: update of row r0 + u
    if (u < 0) {
        // x-face row w (w < nrow) or y-face row w - nrow (up to nrow)
        const bool xdir = w < nrow;
        const int y = w - nrow;
        const bool task = y <= nrow;
        const int k = xdir ? it.r0 + w : it.r0 + y;
        const bool on = task && (xdir ? (j >= it.j0) && (j <= min(it.j0 + STRIP, nx)) : owner);
        double cs = 1.0, sn = 0.0;
        if (!CART && on) {
            const GenG G{B.geom, nx, ny};
            cs = xdir ? G.V(F_c, k, j) : G.H(F_c, k, j);
            sn = xdir ? G.V(F_s, k, j) : G.H(F_s, k, j);
        }
        __syncthreads();
        if (on) {
            const double* const pl = xdir ? sE + w * WG_PLANE + lane - 1 : sN + y * WG_PLANE + lane;
            const double* const pr = xdir ? sW + w * WG_PLANE + lane : sS + y * WG_PLANE + lane;
            Q4 L, Rs;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                L.v[c] = pl[c * WAVE];
                Rs.v[c] = pr[c * WAVE];
            }
            // beyond a side the slot holds the ghost value (outer_state's)
            if (xdir) {
                if (west && j == 0) L = outer_state<CART>(B, PHX_W, Rs, L, k, j);
                if (east && j == nx) Rs = outer_state<CART>(B, PHX_E, L, Rs, k, j);
            } else {
                if (k == 0) L = outer_state<CART>(B, PHX_S, Rs, L, k, j);
                if (k == ny) Rs = outer_state<CART>(B, PHX_N, L, Rs, k - 1, j);
            }
            if (!CART) {
                L = phx::rotate(L, cs, sn);
                Rs = phx::rotate(Rs, cs, sn);
            } else if (!xdir) {
                L = phx::rotate90(L);
                Rs = phx::rotate90(Rs);
            }
            Q4 F = flux_of<FLUX, GEN>(L, Rs, A.ph);
            if (!CART) F = phx::unrotate(F, cs, sn);
            else if (!xdir) F = phx::unrotate90(F);
            double* const pf = (xdir ? fX + w * WG_PLANE : fY + y * WG_PLANE) + lane;
#pragma unroll
            for (int c = 0; c < 4; ++c) pf[c * WAVE] = F.v[c];
        }
        __syncthreads();
        return;
    }
    __syncthreads();
    const bool row = u < nrow;
    const int k = it.r0 + u;
    Q4 pre[EMIT_CHUNK];
    double LW = 0.0, LE = 0.0, LS = 0.0, LN = 0.0, Ac = 1.0, dxc = 0.0;
    const double dt = A.fold_mode == FOLD_DT ? step_dt(A, B.case_id)
                                             : (A.dt != nullptr ? ld_const(A.dt, B.case_id) : 0.0);
    if (row && owner) {
        cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        prefetch_sources(A, B, k, j, pre);
        if (CART && A.dtmin != nullptr) dxc = CartGT<true>{B.geom, nx, ny}.col(C_dx, j);
    }
    __syncthreads();
    if (!row) return;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (owner) {
        Q4 Res;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const double FW = fX[u * WG_PLANE + c * WAVE + lane], FE = fX[u * WG_PLANE + c * WAVE + lane + 1];
            const double FS = fY[u * WG_PLANE + c * WAVE + lane], FN = fY[(u + 1) * WG_PLANE + c * WAVE + lane];
            Res.v[c] = 0.5 * (((LW * (2.0 * FW) - LE * (2.0 * FE)) + LS * (2.0 * FS)) - LN * (2.0 * FN));
        }
        phx::div_all(Res.v, Ac, Res.v);
        emit_row<CART, true>(A, B, k, j, dt, Res, lane_dt, lane_bad, pre, dxc);
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

// CK: geometry kind of the launch's blocks, 0 general, 1 Cartesian, 2 both
template <int CK, int FLUX, int R, bool GEN>
__global__ void __launch_bounds__(wg_waves(R) * WAVE) k_stage_wg(StageArgs A) {
    if (fold_step(A)) return;
    __shared__ double lds[wg_lds(R)];
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride, A.fold_blocks);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) stage_wg_item<true, FLUX, R, GEN>(A, it, lds);
            else stage_wg_item<false, FLUX, R, GEN>(A, it, lds);
        } else {
            stage_wg_item<CK == 1, FLUX, R, GEN>(A, it, lds);
        }
        __syncthreads();  // the next item reuses the exchange buffers
    }
}

// ---------------------------------------------------------------------------------------------
// paired stage: two waves per work item (the fused kernel's strip and rows, one halo row below).
// Wave H reconstructs variables 2H and 2H+1 (the variables of the reconstruction are independent);
// per row the waves exchange through LDS the halves of the face states the other needs (E and W
// go to wave 0, N and S to wave 1), wave 0 evaluates the x-face flux and wave 1 the y-face flux,
// the flux halves are exchanged, and each wave completes the residual and every Butcher output of
// its two variables.  On the last stage of a step wave 1 hands its half of the new state to
// wave 0, which evaluates the CFL quantity and realizability.  Same arithmetic, same association
// order as stage_item: each variable and each face flux is computed exactly as there.  Both waves
// run the same rows, so they reach the same barriers; every LDS slot is written after a barrier
// that follows the other wave's last read of it.
// ---------------------------------------------------------------------------------------------
constexpr int PAIR_WAVES = 2;

struct PairLds {
    double x1[PAIR_WAVES][4][WAVE];  // face-state halves: wave 0 writes N, S (vars 0-1); wave 1 E, W (vars 2-3)
    double x2[PAIR_WAVES][4][WAVE];  // flux halves: wave 0 writes FW, FE (vars 2-3); wave 1 F (vars 0-1)
    double x3[2][WAVE];              // wave 1's half (vars 2-3) of the new state, last stage
};

template <int H>
__device__ __forceinline__ double hv(const Q4& q, int i) { return q.v[2 * H + i]; }

// the two variables of this wave of every output of the stage for cell (kk, j); o = the state
// output's values of these variables
template <bool CART, int H>
__device__ __forceinline__ void emit_half(const StageArgs& A, const DevBlock& B, int kk, int j, double dt,
                                          const double res[2], double o[2]) {
    const long idx = B.off + 4 * ((long)kk * B.nx + j) + 2 * H;
    if (A.Rout) *reinterpret_cast<double2*>(A.Rout + idx) = make_double2(res[0], res[1]);
#pragma unroll 1
    for (int m0 = 0; m0 < A.nout; m0 += EMIT_CHUNK) {
        double2 s[EMIT_CHUNK];
#pragma unroll
        for (int q = 0; q < EMIT_CHUNK; ++q)
            if (m0 + q < A.nout) s[q] = *reinterpret_cast<const double2*>(A.src[m0 + q] + idx);
#pragma unroll
        for (int q = 0; q < EMIT_CHUNK; ++q) {
            const int m = m0 + q;
            if (m >= A.nout) break;
            const double am = A.a[m];
            double2 r = s[q];
            if (am != 0.0) {
                const double cdt = dt * am;  // dt * a[stage][step] (explicit_runge_kutta.py:72)
                r.x = s[q].x + cdt * res[0];
                r.y = s[q].y + cdt * res[1];
            }
            *reinterpret_cast<double2*>(A.dst[m] + idx) = r;
            if (m == A.state_out) { o[0] = r.x; o[1] = r.y; }
        }
    }
}

template <bool CART, int FLUX, bool GEN, int H>
__device__ __forceinline__ void stage_pair_body(const StageArgs& A, const DevItem& it, PairLds& L) {
    const DevBlock& B = it.b;
    const int lane = threadIdx.x & (WAVE - 1);
    const int nx = B.nx, ny = B.ny;
    const int j = it.j0 - HALO + lane;
    const bool valid = (j >= -1) && (j <= nx);
    const bool inner = (j >= 0) && (j < nx);
    const bool gcol = (j == -1) || (j == nx);
    const bool recon = inner && (j >= it.j0 - 1) && (j <= it.j0 + STRIP);
    const bool xface = (j >= it.j0) && (j <= min(it.j0 + STRIP, nx));
    const bool owner = inner && (j >= it.j0) && (j < it.j0 + STRIP);
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    const Phys ph = A.ph;
    const bool cfl = A.dtmin != nullptr && A.state_out >= 0;

    const int kr0 = max(it.r0 - 1, 0);
    const int kr1 = min(it.r1, ny);  // row ny is a virtual row closing the north boundary face

    Q4 Um = phx::q4zero(), Uc = phx::q4zero(), Up = phx::q4zero();
    if (inner) Um = fetch_r<CART, GEN>(A.blocks, B, A.Uin, kr0 - 1, j, ph);
    if (valid) Uc = fetch_r<CART, GEN>(A.blocks, B, A.Uin, kr0, j, ph);

    Q4 QNprev = phx::q4zero();  // wave 1: N state of the previous row
    double part[2] = {0.0, 0.0}, prevLN = 0.0, prevA = 1.0;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;

    for (int k = kr0; k <= kr1; ++k) {
        const bool real = (k < ny);
        if (real) {
            if (inner) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
            else if (gcol && k + 1 <= kr1 && k + 1 < ny) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
        }
        // reconstruction of this wave's two variables
        double e[2] = {0.0, 0.0}, w[2] = {0.0, 0.0}, n[2] = {0.0, 0.0}, s[2] = {0.0, 0.0};
        {
            double uw[2], ue[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                uw[i] = __shfl_up(hv<H>(Uc, i), 1, WAVE);
                ue[i] = __shfl_down(hv<H>(Uc, i), 1, WAVE);
            }
            if (real && recon) {
                const phx::CellGeo g = cell_geo<CART>(B, k, j);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    phx::reconstruct_var<GEN>(hv<H>(Uc, i), uw[i], ue[i], hv<H>(Um, i), hv<H>(Up, i), g, ph.limiter,
                                              e[i], w[i], n[i], s[i]);
            }
        }
        // exchange 1: wave 0 needs E and W of variables 2-3, wave 1 N and S of variables 0-1
        if (H == 0) {
            L.x1[0][0][lane] = n[0]; L.x1[0][1][lane] = n[1];
            L.x1[0][2][lane] = s[0]; L.x1[0][3][lane] = s[1];
        } else {
            L.x1[1][0][lane] = e[0]; L.x1[1][1][lane] = e[1];
            L.x1[1][2][lane] = w[0]; L.x1[1][3][lane] = w[1];
        }
        __syncthreads();
        const bool xrow = (k >= it.r0) && (k < it.r1);
        double fw[2] = {0.0, 0.0}, fe[2] = {0.0, 0.0}, fy[2] = {0.0, 0.0};
        if (H == 0) {
            Q4 rE, rW;
            rE.v[0] = e[0]; rE.v[1] = e[1]; rE.v[2] = L.x1[1][0][lane]; rE.v[3] = L.x1[1][1][lane];
            rW.v[0] = w[0]; rW.v[1] = w[1]; rW.v[2] = L.x1[1][2][lane]; rW.v[3] = L.x1[1][3][lane];
            if (!(real && recon)) rE = rW = phx::q4zero();
            const Q4 qsend = (j == -1) ? Uc : rE;
            const Q4 QEl = shfl_up1(qsend);  // limited east state of cell j-1 (ghost value for j == 0)
            Q4 FW = phx::q4zero();
            if (xrow && xface) {
                const Q4 Lx = (j == 0) ? outer_state<CART>(B, PHX_W, rW, QEl, k, j) : QEl;
                const Q4 Rx = (j == nx) ? outer_state<CART>(B, PHX_E, QEl, Uc, k, j) : rW;
                FW = xflux<CART, FLUX, GEN>(B, Lx, Rx, k, j, ph);
            }
            const Q4 FE = shfl_down1(FW);
            // exchange 2 (write): variables 2-3 of FW and FE for wave 1
            L.x2[0][0][lane] = FW.v[2]; L.x2[0][1][lane] = FW.v[3];
            L.x2[0][2][lane] = FE.v[2]; L.x2[0][3][lane] = FE.v[3];
            fw[0] = FW.v[0]; fw[1] = FW.v[1];
            fe[0] = FE.v[0]; fe[1] = FE.v[1];
        } else {
            Q4 rN, rS;
            rN.v[0] = L.x1[0][0][lane]; rN.v[1] = L.x1[0][1][lane]; rN.v[2] = n[0]; rN.v[3] = n[1];
            rS.v[0] = L.x1[0][2][lane]; rS.v[1] = L.x1[0][3][lane]; rS.v[2] = s[0]; rS.v[3] = s[1];
            if (!(real && recon)) rN = rS = phx::q4zero();
            Q4 F = phx::q4zero();
            if (k >= it.r0 && owner) {
                // face between rows k-1 and k (south face of row k, north face of row k-1)
                const Q4 Ly = (k == 0) ? outer_state<CART>(B, PHX_S, rS, Um, k, j) : QNprev;
                const Q4 Ry = (k == ny) ? outer_state<CART>(B, PHX_N, QNprev, Uc, k - 1, j) : rS;
                F = yflux<CART, FLUX, GEN>(B, Ly, Ry, k, j, ph);
            }
            // exchange 2 (write): variables 0-1 of F for wave 0
            L.x2[1][0][lane] = F.v[0]; L.x2[1][1][lane] = F.v[1];
            fy[0] = F.v[2]; fy[1] = F.v[3];
            QNprev = rN;
        }
        __syncthreads();
        if (H == 0) {
            fy[0] = L.x2[1][0][lane]; fy[1] = L.x2[1][1][lane];
        } else {
            fw[0] = L.x2[0][0][lane]; fw[1] = L.x2[0][1][lane];
            fe[0] = L.x2[0][2][lane]; fe[1] = L.x2[0][3][lane];
        }
        double o[2] = {0.0, 0.0};
        const bool emit = (k >= it.r0) && owner && (k - 1 >= it.r0);
        if (k >= it.r0 && owner) {
            if (emit) {
                // residual of row k-1: 0.5*(W - E + S - N)/A with I = L*(2*F) (fvm/base.py:141-190)
                double res[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) res[i] = 0.5 * (part[i] - prevLN * (2.0 * fy[i]));
                phx::div_all(res, prevA, res);
                emit_half<CART, H>(A, B, k - 1, j, dt, res, o);
            }
            if (xrow) {
                double LW, LE, LS, LN, Ac;
                cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
#pragma unroll
                for (int i = 0; i < 2; ++i) part[i] = (LW * (2.0 * fw[i]) - LE * (2.0 * fe[i])) + LS * (2.0 * fy[i]);
                prevLN = LN;
                prevA = Ac;
            }
        }
        if (cfl) {  // uniform: the new state's CFL quantity and realizability on wave 0
            if (H == 1) { L.x3[0][lane] = o[0]; L.x3[1][lane] = o[1]; }
            __syncthreads();
            if (H == 0 && emit) {
                Q4 q;
                q.v[0] = o[0]; q.v[1] = o[1]; q.v[2] = L.x3[0][lane]; q.v[3] = L.x3[1][lane];
                double dx, dy;
                cell_dxdy<CART>(B, k - 1, j, dx, dy);
                const double t = phx::cell_dt(q, dx, dy, ph);
                if (!(q.v[0] > 0.0) || !(q.v[3] > 0.0) || !(t == t)) lane_bad = true;
                else lane_dt = fmin(lane_dt, t);
            }
        }
        Um = Uc;
        Uc = Up;
    }
    if (H == 0) reduce_item(A, B, lane, lane_dt, lane_bad);
}

template <bool CART, int FLUX, int MINW, bool GEN>
__global__ void __launch_bounds__(PAIR_WAVES * WAVE, MINW) k_stage_pair(StageArgs A) {
    __shared__ PairLds L;
    const int h = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        const DevBlock& B = it.b;
        if (frozen_case(A, B)) continue;  // uniform over the workgroup
        if (h == 0) stage_pair_body<CART, FLUX, GEN, 0>(A, it, L);
        else stage_pair_body<CART, FLUX, GEN, 1>(A, it, L);
        __syncthreads();  // the next item reuses the exchange buffers
    }
}

// ---------------------------------------------------------------------------------------------
// split stage: for small meshes, where short rolling-row items would spend most of their work
// on the halo rows they reconstruct again, the stage runs as three kernels: every cell is
// reconstructed exactly once (k_recon_x, with the x-faces), every y-face flux is evaluated once
// from the stored N/S states (k_yface, one lane per face), then the residual and Butcher updates
// (k_update).  Same arithmetic, same association order as stage_item.
// ---------------------------------------------------------------------------------------------
// k_recon_x: owned columns per wave.  Two halo lanes per side as in the fused kernel: the halo
// cell j0-1 is reconstructed (its E state feeds the W face of the first owned cell) and needs its
// own west neighbour j0-2; likewise on the east side.
constexpr int STRIP_A = WAVE - 2 * HALO;
constexpr int STRIP_B = WAVE;      // k_yface, k_update: no column halo

// ---- nq-point Gauss faces (split stage only; GEN instantiation, nq = A.ph.nq in 2..QMAX) ----
// Face F's sum S_F = sum_i w_i*F_i starting from 0 (integrate_flux, fvm/base.py:168-190); per cell
// the split buffers hold p1 = LW*S_W - LE*S_E, the nq N states then the nq S states
// (8*nq doubles at 2*nq*off + 8*nq*cell) and per y-face S_F.
__device__ __forceinline__ void acc_w(Q4& acc, double w, const Q4& F) {
#pragma unroll
    for (int c = 0; c < 4; ++c) acc.v[c] = acc.v[c] + w * F.v[c];
}

template <bool CART, int FLUX>
__device__ __forceinline__ void recon_x_item_q(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = it.b;
    const int nx = B.nx;
    const int j = it.j0 - HALO + threadIdx.x % WAVE;
    const bool valid = (j >= -1) && (j <= nx);
    const bool inner = (j >= 0) && (j < nx);
    const bool gcol = (j == -1) || (j == nx);
    const bool recon = inner && (j >= it.j0 - 1) && (j <= it.j0 + STRIP_A);
    const bool xface = (j >= it.j0) && (j <= min(it.j0 + STRIP_A, nx));
    const bool owner = inner && (j >= it.j0) && (j < it.j0 + STRIP_A);
    const Phys ph = A.ph;
    const int nq = ph.nq;

    Q4 Um = phx::q4zero(), Uc = phx::q4zero(), Up = phx::q4zero();
    if (inner) Um = fetch_r<CART, true>(A.blocks, B, A.Uin, it.r0 - 1, j, ph);
    if (valid) Uc = fetch_r<CART, true>(A.blocks, B, A.Uin, it.r0, j, ph);
    for (int k = it.r0; k < it.r1; ++k) {
        if (inner) Up = fetch_r<CART, true>(A.blocks, B, A.Uin, k + 1, j, ph);
        else if (gcol && k + 1 < it.r1) Up = fetch_r<CART, true>(A.blocks, B, A.Uin, k + 1, j, ph);
        // the row's loads before its arithmetic: this stage waits for memory half of its time
        phx::CellGeo g;
        phx::QGeo qg;
        double LW = 0.0, LE = 0.0, LS, LN, Ac;
        if (recon) {
            g = cell_geo<CART>(B, k, j);
            qg = cell_qgeo(B, k, j, nq);
        } else {
            for (int f = 0; f < 4; ++f)
                for (int i = 0; i < phx::QMAX; ++i) qg.dx[f][i] = qg.dy[f][i] = 0.0;
        }
        if (owner) cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        if (frozen_case(A, B)) return;
        const Q4 Uw = shift_up1(Uc);
        const Q4 Ue = shift_down1(Uc);
        phx::ReconQ r;
        r.u = r.gx = r.gy = r.phi = phx::q4zero();
        if (recon) r = phx::reconstruct_q(Uc, Uw, Ue, Um, Up, g, qg, nq, ph.limiter);
        Q4 SW = phx::q4zero();  // sum over the W face's points of w_i * F_i
#pragma unroll
        for (int i = 0; i < phx::QMAX; ++i) {
            if (i >= nq) break;
            const Q4 qsend = (j == -1) ? Uc : phx::qstate(r, qg, PHX_E, i);
            const Q4 QEl = shift_up1(qsend);  // limited east state of cell j-1 at point i
            if (xface) {
                const Q4 Wi = phx::qstate(r, qg, PHX_W, i);
                const Q4 L = (j == 0) ? outer_state<CART>(B, PHX_W, Wi, QEl, k, j) : QEl;
                const Q4 R = (j == nx) ? outer_state<CART>(B, PHX_E, QEl, Uc, k, j) : Wi;
                acc_w(SW, phx::gauss_w(nq, i), xflux<CART, FLUX, true>(B, L, R, k, j, ph));
            }
        }
        const Q4 SE = shift_down1(SW);
        if (owner) {
            Q4 part;
#pragma unroll
            for (int c = 0; c < 4; ++c) part.v[c] = LW * SW.v[c] - LE * SE.v[c];
            const long cell = (long)k * nx + j;
            st4(A.p1 + B.off + 4 * cell, part);
            double* sn = A.sn + 2 * nq * B.off + 8 * nq * cell;
#pragma unroll
            for (int i = 0; i < phx::QMAX; ++i) {
                if (i >= nq) break;
                st4(sn + 4 * i, phx::qstate(r, qg, PHX_N, i));
                st4(sn + 4 * (nq + i), phx::qstate(r, qg, PHX_S, i));
            }
        }
        Um = Uc;
        Uc = Up;
    }
}

// Gauss sum S_F = sum_i w_i F_i (from 0) of y-face f of column j
template <bool CART, int FLUX>
__device__ __forceinline__ Q4 yface_sum_q(const StageArgs& A, const DevBlock& B, const double* sn, int f, int j, const Phys& ph) {
    const int nx = B.nx, ny = B.ny;
    const int nq = ph.nq;
    // N states of row f-1 (f > 0) and S states of row f (f < ny)
    const long below = f > 0 ? 8 * nq * ((long)(f - 1) * nx + j) : 0;
    const long above = f < ny ? 8 * nq * ((long)f * nx + j) + 4 * nq : 0;
    Q4 gS = phx::q4zero(), gN = phx::q4zero();
    if (f == 0) gS = fetch_r<CART, true>(A.blocks, B, A.Uin, -1, j, ph);
    if (f == ny) gN = fetch_r<CART, true>(A.blocks, B, A.Uin, ny, j, ph);
    Q4 S = phx::q4zero();
#pragma unroll
    for (int i = 0; i < phx::QMAX; ++i) {
        if (i >= nq) break;
        Q4 L, R;
        if (f == 0) L = outer_state<CART>(B, PHX_S, ld4(sn + above + 4 * i), gS, 0, j);
        else L = ld4(sn + below + 4 * i);
        if (f == ny) R = outer_state<CART>(B, PHX_N, L, gN, ny - 1, j);
        else R = ld4(sn + above + 4 * i);
        acc_w(S, phx::gauss_w(nq, i), yflux<CART, FLUX, true>(B, L, R, f, j, ph));
    }
    return S;
}

template <bool CART, int FLUX>
__device__ __forceinline__ void yface_item_q(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int nx = B.nx;
    const int j = it.j0 + (int)(threadIdx.x % WAVE);
    if (j >= nx) return;
    const double* sn = A.sn + 2 * A.ph.nq * B.off;
    for (int f = it.r0; f < it.r1; ++f)
        st4(A.yf + B.yoff + 4 * ((long)f * nx + j), yface_sum_q<CART, FLUX>(A, B, sn, f, j, A.ph));
}

// Gauss faces, y-faces and update in one pass (variant 5; yface_update_item with the sums S_F)
template <bool CART, int FLUX>
__device__ __forceinline__ void yface_update_item_q(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int nx = B.nx;
    const int j = it.j0 + lane;
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    const Phys ph = A.ph;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (j < nx) {
        const double* sn = A.sn + 2 * ph.nq * B.off;
        Q4 FS = yface_sum_q<CART, FLUX>(A, B, sn, it.r0, j, ph);
        for (int k = it.r0; k < it.r1; ++k) {
            const Q4 FN = yface_sum_q<CART, FLUX>(A, B, sn, k + 1, j, ph);
            const Q4 p = ld4(A.p1 + B.off + 4 * ((long)k * nx + j));
            double LW, LE, LS, LN, Ac;
            cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
            Q4 Res;
#pragma unroll
            for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * FS.v[c]) - LN * FN.v[c]);
            phx::div_all(Res.v, Ac, Res.v);
            emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
            FS = FN;
        }
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void recon_x_item(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = it.b;
    const int nx = B.nx;
    const int j = it.j0 - HALO + threadIdx.x % WAVE;
    const bool valid = (j >= -1) && (j <= nx);
    const bool inner = (j >= 0) && (j < nx);
    const bool gcol = (j == -1) || (j == nx);
    const bool recon = inner && (j >= it.j0 - 1) && (j <= it.j0 + STRIP_A);
    const bool xface = (j >= it.j0) && (j <= min(it.j0 + STRIP_A, nx));
    const bool owner = inner && (j >= it.j0) && (j < it.j0 + STRIP_A);
    const Phys ph = A.ph;

    Q4 Um = phx::q4zero(), Uc = phx::q4zero(), Up = phx::q4zero();
    if (inner) Um = fetch_r<CART, GEN>(A.blocks, B, A.Uin, it.r0 - 1, j, ph);
    if (valid) Uc = fetch_r<CART, GEN>(A.blocks, B, A.Uin, it.r0, j, ph);
    for (int k = it.r0; k < it.r1; ++k) {
        if (inner) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
        else if (gcol && k + 1 < it.r1) Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
        phx::CellGeo g;
        double LW, LE, LS, LN, Ac;
        if (recon) g = cell_geo<CART>(B, k, j);
        if (owner) cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        if (frozen_case(A, B)) return;
        const Q4 Uw = shift_up1(Uc);
        const Q4 Ue = shift_down1(Uc);
        phx::Recon r;
        r.E = r.W = r.N = r.S = phx::q4zero();
        if (recon) {
            r = phx::reconstruct<GEN>(Uc, Uw, Ue, Um, Up, g, ph.limiter);
        }
        const Q4 qsend = (j == -1) ? Uc : r.E;
        const Q4 QEl = shift_up1(qsend);  // limited east state of cell j-1 (ghost value for j == 0)
        Q4 FW = phx::q4zero();
        if (xface) {
            const Q4 L = (j == 0) ? outer_state<CART>(B, PHX_W, r.W, QEl, k, j) : QEl;
            const Q4 R = (j == nx) ? outer_state<CART>(B, PHX_E, QEl, Uc, k, j) : r.W;
            FW = xflux<CART, FLUX, GEN>(B, L, R, k, j, ph);
        }
        const Q4 FE = shift_down1(FW);
        if (owner) {
            Q4 part;
#pragma unroll
            for (int c = 0; c < 4; ++c) part.v[c] = LW * (2.0 * FW.v[c]) - LE * (2.0 * FE.v[c]);
            const long cell = (long)k * nx + j;
            st4(A.p1 + B.off + 4 * cell, part);
            st4(A.sn + 2 * B.off + 8 * cell, r.N);
            st4(A.sn + 2 * B.off + 8 * cell + 4, r.S);
        }
        Um = Uc;
        Uc = Up;
    }
}

// y-faces of face rows [r0, r1) of a strip of 64 columns (face f between rows f-1 and f; f = 0 and
// f = ny take the outer states of the S and N boundaries): one flux per lane and face, stored.
template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void yface_item(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int nx = B.nx, ny = B.ny;
    const int j = it.j0 + (int)(threadIdx.x % WAVE);
    if (j >= nx) return;
    const Phys ph = A.ph;
    const double* sn = A.sn + 2 * B.off;
    for (int f = it.r0; f < it.r1; ++f) {
        Q4 L, R;
        if (f == 0) L = outer_state<CART>(B, PHX_S, ld4(sn + 8 * (long)j + 4), fetch_r<CART, GEN>(A.blocks, B, A.Uin, -1, j, ph), 0, j);
        else L = ld4(sn + 8 * ((long)(f - 1) * nx + j));
        if (f == ny) R = outer_state<CART>(B, PHX_N, L, fetch_r<CART, GEN>(A.blocks, B, A.Uin, ny, j, ph), ny - 1, j);
        else R = ld4(sn + 8 * ((long)f * nx + j) + 4);
        st4(A.yf + B.yoff + 4 * ((long)f * nx + j), yflux<CART, FLUX, GEN>(B, L, R, f, j, ph));
    }
}

// residual ((x-part + LS*(2 F_S)) - LN*(2 F_N))/A (Gauss sums S_F in place of 2 F with nq > 1) of rows [r0, r1) of a 64-column strip, then every
// Butcher output, the CFL quantity and realizability (as the fused kernel).
template <bool CART>
__device__ __forceinline__ void update_item(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int nx = B.nx;
    const int j = it.j0 + lane;
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (j < nx) {
        const double* yf = A.yf + B.yoff + 4 * (long)j;
        Q4 FS = ld4(yf + 4 * (long)it.r0 * nx);
        for (int k = it.r0; k < it.r1; ++k) {
            const Q4 FN = ld4(yf + 4 * (long)(k + 1) * nx);
            const Q4 p = ld4(A.p1 + B.off + 4 * ((long)k * nx + j));
            double LW, LE, LS, LN, Ac;
            cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
            Q4 Res;
            if (A.ph.nq > 1) {  // y-face entries are the Gauss sums already
#pragma unroll
                for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * FS.v[c]) - LN * FN.v[c]);
                phx::div_all(Res.v, Ac, Res.v);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * (2.0 * FS.v[c])) - LN * (2.0 * FN.v[c]));
                phx::div_all(Res.v, Ac, Res.v);
            }
            emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
            FS = FN;
        }
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

// y-faces and update in one pass (variant 5): the lane of column j walks the face rows of cell
// rows [r0, r1); after the flux of face k+1 it has both y-fluxes of cell (k, j) and completes its
// residual and Butcher outputs as update_item does.  Face r0 is evaluated again by the item
// below (one extra flux per item and column instead of a y-flux buffer and a third kernel).
template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ Q4 yface_flux_at(const StageArgs& A, const DevBlock& B, const double* sn, int f, int j,
                                            const Phys& ph) {
    const int nx = B.nx, ny = B.ny;
    Q4 L, R;
    if (f == 0) L = outer_state<CART>(B, PHX_S, ld4(sn + 8 * (long)j + 4), fetch_r<CART, GEN>(A.blocks, B, A.Uin, -1, j, ph), 0, j);
    else L = ld4(sn + 8 * ((long)(f - 1) * nx + j));
    if (f == ny) R = outer_state<CART>(B, PHX_N, L, fetch_r<CART, GEN>(A.blocks, B, A.Uin, ny, j, ph), ny - 1, j);
    else R = ld4(sn + 8 * ((long)f * nx + j) + 4);
    return yflux<CART, FLUX, GEN>(B, L, R, f, j, ph);
}

template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void yface_update_item(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int nx = B.nx;
    const int j = it.j0 + lane;
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    const Phys ph = A.ph;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (j < nx) {
        const double* sn = A.sn + 2 * B.off;
        Q4 FS = yface_flux_at<CART, FLUX, GEN>(A, B, sn, it.r0, j, ph);
        for (int k = it.r0; k < it.r1; ++k) {
            const Q4 FN = yface_flux_at<CART, FLUX, GEN>(A, B, sn, k + 1, j, ph);
            const Q4 p = ld4(A.p1 + B.off + 4 * ((long)k * nx + j));
            double LW, LE, LS, LN, Ac;
            cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
            Q4 Res;
#pragma unroll
            for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * (2.0 * FS.v[c])) - LN * (2.0 * FN.v[c]));
            phx::div_all(Res.v, Ac, Res.v);
            emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
            FS = FN;
        }
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

// y-faces and update with one face per wave (variant 6): a workgroup of R+1 waves takes R cell rows
// [r0, r1) of a 64-column strip; wave w evaluates face r0+w into LDS, and after one barrier wave w < R
// completes cell row r0+w from faces r0+w and r0+w+1 as update_item does.  Every wave's chain is one
// flux and at most one update, and a face is evaluated twice only at item boundaries.
constexpr int YU_MAX_ROWS = 7;  // rows per item (R + 1 <= 8 waves per workgroup)

// Q = true: Gauss faces (the sums S_F of yface_sum_q, the residual of the nq-point rule)
template <bool CART, int FLUX, bool GEN, bool Q>
__device__ __forceinline__ void yface_update_wg_item(const StageArgs& A, const DevItem& it, Q4* lds) {
    const DevBlock B = it.b;  // in scalar registers
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = threadIdx.x / WAVE;
    const int nx = B.nx;
    const int j = it.j0 + lane;
    const int nrow = it.r1 - it.r0;
    const Phys ph = A.ph;
    const bool dead = frozen_case(A, B);
    if (dead) return;  // uniform over the workgroup
    if (w <= nrow && j < nx) {
        if (Q) lds[w * WAVE + lane] = yface_sum_q<CART, FLUX>(A, B, A.sn + 2 * ph.nq * B.off, it.r0 + w, j, ph);
        else lds[w * WAVE + lane] = yface_flux_at<CART, FLUX, GEN>(A, B, A.sn + 2 * B.off, it.r0 + w, j, ph);
    }
    __syncthreads();
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (w < nrow && j < nx) {
        const int k = it.r0 + w;
        const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
        const Q4 FS = lds[w * WAVE + lane], FN = lds[(w + 1) * WAVE + lane];
        const Q4 p = ld4(A.p1 + B.off + 4 * ((long)k * nx + j));
        double LW, LE, LS, LN, Ac;
        cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        Q4 Res;
        if (Q) {  // the face entries are the Gauss sums already
#pragma unroll
            for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * FS.v[c]) - LN * FN.v[c]);
            phx::div_all(Res.v, Ac, Res.v);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) Res.v[c] = 0.5 * ((p.v[c] + LS * (2.0 * FS.v[c])) - LN * (2.0 * FN.v[c]));
            phx::div_all(Res.v, Ac, Res.v);
        }
        emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

// CK: geometry kind of the launch's blocks, 0 general, 1 Cartesian, 2 both (the path chosen per
// item's block; one launch over the merged list of a mesh with both kinds)
template <int CK, int FLUX, bool GEN, bool Q>
__global__ void __launch_bounds__((YU_MAX_ROWS + 1) * WAVE) k_yface_update_wg(StageArgs A) {
    __shared__ Q4 lds[(YU_MAX_ROWS + 1) * WAVE];
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) yface_update_wg_item<true, FLUX, GEN, Q>(A, it, lds);
            else yface_update_wg_item<false, FLUX, GEN, Q>(A, it, lds);
        } else {
            yface_update_wg_item<CK == 1, FLUX, GEN, Q>(A, it, lds);
        }
        __syncthreads();  // the next item reuses the face buffer
    }
}

// y-faces and update over flat cell ranges (variant 8): a workgroup of T lanes takes the cells
// c in [c0, c0 + n) of one block in row-major order.  The S face of cell c has the face index c and
// its N face c + nx (face (f, j) at f*nx + j, f = 0..ny), so the faces of the range are the n + nx
// consecutive indices from c0: lane t evaluates faces c0 + t, c0 + t + T, ... into LDS and, after
// one barrier, completes cells c0 + t, c0 + t + T, ... as update_item does.  No lane idles on a
// partial column strip, and a face is evaluated twice only where two ranges meet (nx faces per
// range).  T = (A.rows_wave + 1) * WAVE; the host sizes the ranges so that n + nx <= A.fq * T, the
// faces the dynamic LDS holds.
template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void yface_update_flat_item(const StageArgs& A, const DevItem& it, Q4* lds) {
    const DevBlock B = it.b;  // in scalar registers
    if (frozen_case(A, B)) return;  // uniform over the workgroup
    const int T = blockDim.x;
    const int t = threadIdx.x;
    const int lane = t & (WAVE - 1);
    const int nx = B.nx;
    const int c0 = it.j0, n = it.r0;
    const Phys ph = A.ph;
    const double* sn = A.sn + 2 * B.off;
    for (int q = t; q < n + nx; q += T) {
        const int fi = c0 + q;
        const int f = fi / nx;
        lds[q] = yface_flux_at<CART, FLUX, GEN>(A, B, sn, f, fi - f * nx, ph);
    }
    __syncthreads();
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
    for (int q = t; q < n; q += T) {
        const int c = c0 + q;
        const int k = c / nx, j = c - k * nx;
        const Q4 FS = lds[q], FN = lds[q + nx];
        const Q4 p = ld4(A.p1 + B.off + 4 * (long)c);
        double LW, LE, LS, LN, Ac;
        cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
        Q4 Res;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) Res.v[cc] = 0.5 * ((p.v[cc] + LS * (2.0 * FS.v[cc])) - LN * (2.0 * FN.v[cc]));
        phx::div_all(Res.v, Ac, Res.v);
        emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
    }
    reduce_item(A, B, lane, lane_dt, lane_bad);
}

constexpr int FLAT_MAX_WAVES = 16;  // workgroup of up to 1024 lanes

template <bool CART, int FLUX, bool GEN>
__global__ void __launch_bounds__(FLAT_MAX_WAVES * WAVE) k_yface_update_flat(StageArgs A) {
    extern __shared__ Q4 flat_lds[];
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) {
        yface_update_flat_item<CART, FLUX, GEN>(A, const_ref(A.items, i), flat_lds);
        __syncthreads();  // the next item reuses the face buffer
    }
}

template <bool CART, int FLUX, bool GEN>
__global__ void __launch_bounds__(WAVE) k_yface_update(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) yface_update_item<CART, FLUX, GEN>(A, const_ref(A.items, i));
}

template <int CK, int FLUX, int MINW, bool GEN>
__global__ void __launch_bounds__(WAVE, MINW) k_recon_x(StageArgs A) {
    if (fold_step(A)) return;
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride, A.fold_blocks);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) recon_x_item<true, FLUX, GEN>(A, it);
            else recon_x_item<false, FLUX, GEN>(A, it);
        } else {
            recon_x_item<CK == 1, FLUX, GEN>(A, it);
        }
    }
}

// k_recon_x_lin: the reconstruction kernel of the split stage over the row-major positions of a
// block, p = k*(nx+1) + j with j in [0, nx]: j < nx is cell (k, j) and its west face, j = nx the
// east boundary face of row k.  Lane l of an item takes position j0 - 1 + l; lane 0 only
// reconstructs (its limited east state feeds the west face of lane 1), lane WAVE-1 only evaluates
// its face (the east face flux of lane WAVE-2), lanes 1..WAVE-2 own their positions.  East and west
// neighbour values come from the adjacent lanes inside a row and from memory at row ends and at the
// wave's two edge lanes.  Rows that are not a multiple of a column strip leave no idle lanes, and
// each wave needs one halo lane per side instead of two.  Same arithmetic and association order as
// recon_x_item.
constexpr int LIN_OWN = WAVE - 2;

template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void recon_x_lin_item(const StageArgs& A, const DevItem& it) {
    const DevBlock B = it.b;  // in scalar registers
    const int nx = B.nx, npos = B.ny * (nx + 1);
    const int lane = threadIdx.x % WAVE;
    const int p = it.j0 - 1 + lane;
    const bool valid = (p >= 0) && (p < npos);
    const int k = valid ? p / (nx + 1) : 0;
    const int j = valid ? p - k * (nx + 1) : 0;
    const bool cell = valid && (j < nx);
    const Phys ph = A.ph;

    // every load is issued before the first shuffle, so that a wave waits for memory once
    const bool wmem = cell && (j == 0 || lane == 0);
    const bool emem = cell && (lane == WAVE - 1);
    Q4 Uc = phx::q4zero(), Um = phx::q4zero(), Up = phx::q4zero(), Uw = phx::q4zero(), Ue = phx::q4zero();
    if (valid) Uc = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k, j, ph);  // j == nx: the east ghost value
    if (cell) {
        Um = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k - 1, j, ph);
        Up = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k + 1, j, ph);
    }
    if (wmem) Uw = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k, j - 1, ph);
    if (emem) Ue = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k, j + 1, ph);
    phx::CellGeo g;
    double LW, LE, LS, LN, Ac;
    if (cell) {
        g = cell_geo<CART>(B, k, j);
        cell_L<CART>(B, k, j, LW, LE, LS, LN, Ac);
    }
    if (frozen_case(A, B)) return;
    const Q4 Uwl = shift_up1(Uc);
    const Q4 Uel = shift_down1(Uc);
    if (!wmem) Uw = Uwl;
    if (!emem) Ue = Uel;
    phx::Recon r;
    r.E = r.W = r.N = r.S = phx::q4zero();
    if (cell) {
        r = phx::reconstruct<GEN>(Uc, Uw, Ue, Um, Up, g, ph.limiter);
    }
    const Q4 QEl = shift_up1(r.E);  // limited east state of position p-1 (cell j-1 of the same row for j > 0)
    Q4 FW = phx::q4zero();
    if (valid && lane > 0) {
        const Q4 L = (j == 0) ? outer_state<CART>(B, PHX_W, r.W, Uw, k, j) : QEl;
        const Q4 R = (j == nx) ? outer_state<CART>(B, PHX_E, QEl, Uc, k, j) : r.W;
        FW = xflux<CART, FLUX, GEN>(B, L, R, k, j, ph);
    }
    const Q4 FE = shift_down1(FW);
    if (cell && lane > 0 && lane < WAVE - 1) {
        Q4 part;
#pragma unroll
        for (int c = 0; c < 4; ++c) part.v[c] = LW * (2.0 * FW.v[c]) - LE * (2.0 * FE.v[c]);
        const long cidx = (long)k * nx + j;
        st4(A.p1 + B.off + 4 * cidx, part);
        st4(A.sn + 2 * B.off + 8 * cidx, r.N);
        st4(A.sn + 2 * B.off + 8 * cidx + 4, r.S);
    }
}

template <int CK, int FLUX, int MINW, bool GEN>
__global__ void __launch_bounds__(WAVE, MINW) k_recon_x_lin(StageArgs A) {
    if (fold_step(A)) return;
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride, A.fold_blocks);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) recon_x_lin_item<true, FLUX, GEN>(A, it);
            else recon_x_lin_item<false, FLUX, GEN>(A, it);
        } else {
            recon_x_lin_item<CK == 1, FLUX, GEN>(A, it);
        }
    }
}

template <bool CART, int FLUX, bool GEN>
__global__ void __launch_bounds__(WAVE) k_yface(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) yface_item<CART, FLUX, GEN>(A, const_ref(A.items, i));
}

// Gauss faces (nq > 1): kernels of their own, so that the register budget of the 1-point kernels is
// not set by the nq-point path
template <bool CART, int FLUX>
__global__ void __launch_bounds__(WAVE, 2) k_recon_x_q(StageArgs A) {
    if (fold_step(A)) return;
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride, A.fold_blocks);
    for (int i = first; i < hi; i += stride) recon_x_item_q<CART, FLUX>(A, const_ref(A.items, i));
}

template <bool CART, int FLUX>
__global__ void __launch_bounds__(WAVE) k_yface_q(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) yface_item_q<CART, FLUX>(A, const_ref(A.items, i));
}

template <bool CART, int FLUX>
__global__ void __launch_bounds__(WAVE) k_yface_update_q(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) yface_update_item_q<CART, FLUX>(A, const_ref(A.items, i));
}

template <bool CART>
__global__ void __launch_bounds__(WAVE) k_update(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) update_item<CART>(A, const_ref(A.items, i));
}

// ---------------------------------------------------------------------------------------------
// element-wise stage (small meshes, where one lane per cell leaves most SIMDs with one or two
// waves): the same arithmetic as stage_item in three passes with more lanes in flight,
//   k_ew_recon   one lane per cell and variable: limited face states E, W, N, S (the variables of
//                the reconstruction are independent: reconstruct_var)
//   k_ew_face    one lane per face: left/right states (block-edge faces: outer state) -> flux
//   k_ew_update  one lane per cell: residual, every Butcher output, CFL quantity, realizability
// Tiles {block, first element, count}: EW_WG / 4 cells, EW_WG faces, EW_WG cells.  Cells are numbered
// k*nx + j in their block; faces as in the adjoint (x-faces (k, jf) first, then y-faces (kf, j)).
// ---------------------------------------------------------------------------------------------
constexpr int EW_WG = 256;
constexpr int EW_RCELLS = EW_WG / 4;

// variable v of cell (k, j) (one cell outside the block at most, never a corner), in the
// reconstruction variables; own cells are read directly, ghosts through fetch_r
template <bool CART, bool GEN>
__device__ __forceinline__ double ew_value(const StageArgs& A, const DevBlock& B, int k, int j, int v,
                                           const Phys& ph) {
    if (!(GEN && ph.prim) && k >= 0 && k < B.ny && j >= 0 && j < B.nx)
        return gld(A.Uin, B.off + 4 * ((long)k * B.nx + j) + v);
    const Q4 q = fetch_r<CART, GEN>(A.blocks, B, A.Uin, k, j, ph);
    return v == 0 ? q.v[0] : (v == 1 ? q.v[1] : (v == 2 ? q.v[2] : q.v[3]));
}

template <bool CART, bool GEN>
__device__ __forceinline__ void ew_recon_tile(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    const int c = (int)threadIdx.x >> 2, v = (int)threadIdx.x & 3;
    if (c >= it.r0) return;
    const int e = it.j0 + c;
    const int k = e / B.nx, j = e - k * B.nx;
    const Phys ph = A.ph;
    const double u = ew_value<CART, GEN>(A, B, k, j, v, ph);
    const double uw = ew_value<CART, GEN>(A, B, k, j - 1, v, ph);
    const double ue = ew_value<CART, GEN>(A, B, k, j + 1, v, ph);
    const double us = ew_value<CART, GEN>(A, B, k - 1, j, v, ph);
    const double un = ew_value<CART, GEN>(A, B, k + 1, j, v, ph);
    const phx::CellGeo g = cell_geo<CART>(B, k, j);
    double qE, qW, qN, qS;
    phx::reconstruct_var<GEN>(u, uw, ue, us, un, g, ph.limiter, qE, qW, qN, qS);
    double* rb = A.rb + phx::adj::RB * (B.off / 4 + e) + v;
    rb[phx::adj::RB_E] = qE;
    rb[phx::adj::RB_W] = qW;
    rb[phx::adj::RB_N] = qN;
    rb[phx::adj::RB_S] = qS;
}

template <bool CART, int FLUX, bool GEN>
__device__ __forceinline__ void ew_face_tile(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;
    if ((int)threadIdx.x >= it.r0) return;
    const long long f = (long long)it.j0 + threadIdx.x;
    const phx::host::AdjBlock O{B.off / 4, B.foff};
    const phx::adj::FaceRef F = phx::adj::face_ref(B, f);
    Q4 L, R;
    phx::adj::face_states<CART>(A.blocks, B, A.Uin, A.rb, O, F, L, R, A.ph);
    const Q4 Fl = F.xdir ? xflux<CART, FLUX, GEN>(B, L, R, F.k, F.j, A.ph)
                         : yflux<CART, FLUX, GEN>(B, L, R, F.k, F.j, A.ph);
    st4(A.ff + 4 * (B.foff + f), Fl);
}

template <bool CART>
__device__ __forceinline__ void ew_update_tile(const StageArgs& A, const DevItem& it) {
    const DevBlock& B = A.blocks[it.block];
    if (frozen_case(A, B)) return;  // uniform over the workgroup
    const int t = (int)threadIdx.x;
    double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
    bool lane_bad = false;
    if (t < it.r0) {
        const int e = it.j0 + t;
        const int k = e / B.nx, j = e - k * B.nx;
        const phx::host::AdjBlock O{B.off / 4, B.foff};
        const Q4 Res = phx::adj::cell_residual<CART>(B, O, A.ff, k, j);
        const double dt = (A.dt != nullptr) ? ld_const(A.dt, B.case_id) : 0.0;
        emit_row<CART>(A, B, k, j, dt, Res, lane_dt, lane_bad);
    }
    reduce_item(A, B, t & (WAVE - 1), lane_dt, lane_bad);  // every lane of the wave takes part
}

template <int CK, bool GEN>
__global__ void __launch_bounds__(EW_WG) k_ew_recon(StageArgs A) {
    if (fold_step(A)) return;
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride, A.fold_blocks);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {  // items of both geometry kinds: the path of the item's block
            if (it.b.kind == PHX_GEOM_CARTESIAN) ew_recon_tile<true, GEN>(A, it);
            else ew_recon_tile<false, GEN>(A, it);
        } else {
            ew_recon_tile<CK == 1, GEN>(A, it);
        }
    }
}

template <int CK, int FLUX, bool GEN>
__global__ void __launch_bounds__(EW_WG) k_ew_face(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) ew_face_tile<true, FLUX, GEN>(A, it);
            else ew_face_tile<false, FLUX, GEN>(A, it);
        } else {
            ew_face_tile<CK == 1, FLUX, GEN>(A, it);
        }
    }
}

template <int CK>
__global__ void __launch_bounds__(EW_WG) k_ew_update(StageArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        if (CK == 2) {
            if (it.b.kind == PHX_GEOM_CARTESIAN) ew_update_tile<true>(A, it);
            else ew_update_tile<false>(A, it);
        } else {
            ew_update_tile<CK == 1>(A, it);
        }
    }
}

// Launchers of the stage kernel families, one per kernel template; each is defined in the translation
// unit that instantiates its kernels (the instances take minutes to compile, so they are spread over
// several units).  kind: 1 Cartesian, 0 general blocks; minw = register budget asked for (2, 3 or 4), which
// each launcher turns into the waves per SIMD of its instances, those that compile without heavy
// spilling: fused and paired 2-3 (2 generic), strip reconstruction 2-3 (2 generic), row-major
// reconstruction 3-4 (4 with HLLL, 3 generic); the y-face and update kernels need no limiter and are
// built once.
struct k_stage_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_stage_wg_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_stage_pair_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_recon_x_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_recon_x_lin_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_recon_x_q_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_q_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_ew_recon_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_ew_face_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_ew_update_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_update_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_update_q_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_update_wg_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_update_wg_q_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_yface_update_flat_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
struct k_update_tag {
    static void launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A);
};
// The same over the merged list of both geometry kinds (the path chosen per item's block): one launch
// of phase p (0 reconstruction, 1 faces, 2 update) of the element-wise stage, of the reconstruction of
// variants 6 and 7, and of the y-face and update kernel of variants 6 and 7.
void launch_ew_mixed(const phx_plan* P, StageArgs A, int p, hipStream_t st);
void launch_stage_wg_mixed(const phx_plan* P, StageArgs A, hipStream_t st);
void launch_recon_x_mixed(const phx_plan* P, StageArgs A, hipStream_t st);
void launch_recon_x_lin_mixed(const phx_plan* P, StageArgs A, hipStream_t st);
void launch_yface_wg_mixed(const phx_plan* P, StageArgs A, hipStream_t st);

// the generic instantiation: another limiter, primitive-variable reconstruction or Gauss faces
inline bool generic_instance(const phx_plan* P) {
    return P->ph.limiter != PHX_LIMITER_VENKATAKRISHNAN || P->ph.prim || P->ph.nq > 1;
}

// T::go<Cartesian, flux, waves per SIMD, generic> for the plan's flux and options
template <class T>
void dispatch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    const bool roe = P->flux == PHX_FLUX_ROE;
    const bool gen = generic_instance(P);
#define PHX_LAUNCH_M(C, F)                                                                       \
    do {                                                                                         \
        if (gen) T::template go<C, F, 2, true>(g, st, A);                                        \
        else if (minw == 4) T::template go<C, F, 4, false>(g, st, A);                            \
        else if (minw == 3) T::template go<C, F, 3, false>(g, st, A);                            \
        else T::template go<C, F, 2, false>(g, st, A);                                           \
    } while (0)
    if (kind == 1) {
        if (roe) PHX_LAUNCH_M(true, 0);
        else PHX_LAUNCH_M(true, 1);
    } else {
        if (roe) PHX_LAUNCH_M(false, 0);
        else PHX_LAUNCH_M(false, 1);
    }
#undef PHX_LAUNCH_M
}

}  // namespace stage
}  // namespace phx
