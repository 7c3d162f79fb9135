// phx_kernels.hip -- the stage loop, plans and the C ABI declared in include/pyhype_hip.h, with the small
// kernels (time step, ghosts, resets); the stage kernels are in phx_stage.hpp.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "phx_stage.hpp"

using phx::Phys;
using phx::Q4;
using namespace phx::dev;
using namespace phx::host;
using namespace phx::stage;

namespace {

// Step graphs of phx_run: graph g holds 2^g steps.
constexpr int GRAPHS = phx_plan::GRAPHS;
int dt_slots_for(int ncases) {
    int n = DT_SLOTS;
    while (n > 4 && (long)n * ncases > 256) n >>= 1;
    return n;
}

// standalone CFL reduction over the owned cells of every work item
struct DtArgs {
    const DevItem* items;
    int nitems;
    int strip;  // owned columns per item of this work list
    const double* U;
    unsigned long long* dtmin;
    int* bad;
    const int* step;
    int nslot;
    Phys ph;
};

template <bool CART>
__global__ void __launch_bounds__(WAVE) k_dt(DtArgs A) {
    int lo, hi, first, stride;
    item_range(A.nitems, lo, hi, first, stride);
    const int lane = threadIdx.x & (WAVE - 1);
    for (int i = first; i < hi; i += stride) {
        const DevItem& it = const_ref(A.items, i);
        const DevBlock& B = it.b;
        const int j = it.j0 + lane;
        const bool own = (lane < A.strip) && (j < B.nx);
        double lane_dt = __longlong_as_double((long long)DT_INF_BITS);
        bool lane_bad = false;
        if (own) {
            for (int k = it.r0; k < it.r1; ++k) {
                const Q4 q = ld4(A.U + B.off + 4 * ((long)k * B.nx + j));
                double dx, dy;
                cell_dxdy<CART>(B, k, j, dx, dy);
                const double t = phx::cell_dt(q, dx, dy, A.ph);
                if (!(q.v[0] > 0.0) || !(q.v[3] > 0.0) || !(t == t)) lane_bad = true;
                else lane_dt = fmin(lane_dt, t);
            }
        }
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

// dt = CFL*min, clipped to t_final - t (solvers/base.py:126-136); advance t (Euler2D.py:209).
// One workgroup; a case that failed at an earlier step gets dt = 0 and keeps its time.
// One lane per slot (nslot lanes per case, one memory round trip), the minima combined by shuffles
// inside the lane group; slots cleared when advancing.  The case loop bound is uniform, so every
// lane takes part in the shuffles.  Launched as one workgroup of FIN_THREADS threads.
constexpr int FIN_THREADS = 1024;
__global__ void __launch_bounds__(FIN_THREADS) k_finalize(int ncases, int nslot, double cfl, unsigned long long* dtmin,
                                                          const double* tfinal, double* t, double* dt, int* step,
                                                          const int* bad, const double* frozen, int advance) {
    const int s_next = step[0] + 1;
    const int g = threadIdx.x & (nslot - 1);
    const int per_pass = blockDim.x / nslot;
    for (int base = 0; base < ncases; base += per_pass) {
        const int c = base + threadIdx.x / nslot;
        const bool active = c < ncases;
        unsigned long long m = DT_INF_BITS;
        if (active && frozen == nullptr) m = dtmin[dt_slot(c, g, nslot)];
        for (int o = nslot / 2; o > 0; o >>= 1) {
            const unsigned long long x = __shfl_xor(m, o, nslot);
            m = x < m ? x : m;
        }
        if (!active) continue;
        if (advance) dtmin[dt_slot(c, g, nslot)] = DT_INF_BITS;
        if (g != 0) continue;
        double d;
        if (frozen != nullptr) {
            d = frozen[c];
        } else {
            d = cfl * __longlong_as_double((long long)m);
            const double rem = tfinal[c] - t[c];
            if (rem < d) d = rem;
        }
        if (advance && bad[c] < s_next) d = 0.0;
        dt[c] = d;
        if (advance) t[c] = t[c] + d;
    }
    __syncthreads();
    if (advance && threadIdx.x == 0) step[0] = s_next;
}
// start times of cases [c0, c0 + RESET_CASES), by value: no buffer, copy or wait for one
constexpr int RESET_CASES = 64;
struct StartTimes {
    double t[RESET_CASES];
};
__global__ void k_reset(int ncases, int nslot, int c0, StartTimes T, double* t, unsigned long long* dtmin, int* bad,
                        int* step, int step0) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;  // one thread per (set, case, slot)
    if (c0 == 0) {
        if (c < 2 * ncases * nslot) dtmin[(long)c * DT_STRIDE] = DT_INF_BITS;
        if (c == 0) step[0] = step0;
    }
    if (c < RESET_CASES && c0 + c < ncases) {
        t[c0 + c] = T.t[c];
        bad[c0 + c] = NEVER;
    }
}

__global__ void k_fill_inf(int ncases, int nslot, unsigned long long* dtmin) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;  // one thread per (case, slot)
    if (i < ncases * nslot) dtmin[(long)i * DT_STRIDE] = DT_INF_BITS;
}

// ghost strips for tests: block b, cell index i over E(ny) W(ny) N(nx) S(nx)
__global__ void k_ghosts(const DevBlock* blocks, int nblocks, const long long* goff, const double* U, double* G) {
    const int b = blockIdx.x;
    if (b >= nblocks) return;
    const DevBlock& B = blocks[b];
    const int n = 2 * B.ny + 2 * B.nx;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        int k, j;
        if (i < B.ny) { k = i; j = B.nx; }
        else if (i < 2 * B.ny) { k = i - B.ny; j = -1; }
        else if (i < 2 * B.ny + B.nx) { k = B.ny; j = i - 2 * B.ny; }
        else { k = -1; j = i - 2 * B.ny - B.nx; }
        const Q4 q = (B.kind == PHX_GEOM_CARTESIAN) ? fetch<true>(blocks, B, U, k, j) : fetch<false>(blocks, B, U, k, j);
        st4(G + goff[b] + 4L * i, q);
    }
}

}  // namespace

// =============================================================================================
// host side
// =============================================================================================
namespace {
thread_local std::string g_err;
}  // namespace

int phx::host::fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

namespace {

double* buf_ptr(phx_plan* P, double* U, int id) {
    if (id == BUF_USER) return U;
    if (id == BUF_S0) return P->sbuf[0];
    if (id == BUF_S1) return P->sbuf[1];
    return P->acc[id - BUF_ACC0];
}

// Butcher table -> per-stage program in accumulator form: U^(s+1) = P_s + (dt a_ss) k_s and
// P_t += (dt a_ts) k_s for later rows t, each P_t starting from U0; zero coefficients skipped,
// which reproduces the summation order of ExplicitRungeKutta.integrate (explicit_runge_kutta.py:63-75).
int build_programs(phx_plan* P, int S, const double* a) {
    std::vector<int> Pt(S, BUF_USER);
    std::vector<int> free_acc;
    int nacc = 0;
    P->progs.clear();
    for (int s = 0; s < S; ++s) {
        StageProg g;
        g.in = (s == 0) ? BUF_USER : ((s - 1) % 2 == 0 ? BUF_S0 : BUF_S1);
        // the last stage writes the caller's state in place unless it also reads it as stencil input
        const int out = (s == S - 1 && S > 1) ? BUF_USER : (s % 2 == 0 ? BUF_S0 : BUF_S1);
        g.outs.push_back({out, Pt[s], a[s * S + s]});
        g.state_out = (s == S - 1) ? 0 : -1;
        if (Pt[s] >= BUF_ACC0) free_acc.push_back(Pt[s]);
        for (int t = s + 1; t < S; ++t) {
            const double c = a[t * S + s];
            if (c == 0.0) continue;
            if (Pt[t] == BUF_USER) {
                int id;
                if (!free_acc.empty()) { id = free_acc.back(); free_acc.pop_back(); }
                else { if (nacc >= MAX_ACC) return fail(PHX_E_INVALID, "Butcher table needs too many accumulators"); id = BUF_ACC0 + nacc++; }
                g.outs.push_back({id, BUF_USER, c});
                Pt[t] = id;
            } else {
                g.outs.push_back({Pt[t], Pt[t], c});
            }
        }
        if ((int)g.outs.size() > MAX_OUT) return fail(PHX_E_INVALID, "Butcher stage has too many outputs");
        P->progs.push_back(g);
    }
    P->nacc = nacc;
    P->copy_back = (S == 1);
    return PHX_OK;
}

// a work list on the device, each item with its block's descriptor
int upload_list(const phx_plan* P, const std::vector<WorkItem>& items, DevItem*& dev) {
    if (items.empty()) return PHX_OK;
    std::vector<DevItem> full(items.size());
    for (size_t i = 0; i < items.size(); ++i)
        full[i] = DevItem{items[i].block, items[i].j0, items[i].r0, items[i].r1, P->hblocks[items[i].block]};
    PHX_CK(hipMalloc(&dev, full.size() * sizeof(DevItem)));
    PHX_CK(hipMemcpy(dev, full.data(), full.size() * sizeof(DevItem), hipMemcpyHostToDevice));
    return PHX_OK;
}

int upload_items(const phx_plan* P, std::vector<WorkItem> (&items)[2], DevItem* (&ditems)[2], int (&grid)[2],
                 int grid_waves) {
    for (int kind = 0; kind < 2; ++kind) {
        const size_t n = items[kind].size();
        const int rc = upload_list(P, items[kind], ditems[kind]);
        if (rc) return rc;
        grid[kind] = (int)((grid_waves > 0 && (size_t)grid_waves < n) ? grid_waves : n);
    }
    return PHX_OK;
}

// Whether a block's geometry has an entry beyond 2^60 in magnitude (or not finite) or an area below
// 2^-60: the range for which the limiter's in-range divisions are proven (limit_venkat).
bool odd_geometry(const phx_block_desc& d) {
    for (int64_t i = 0; i < d.geom_len; ++i)
        if (!(fabs(d.geom[i]) <= 0x1p60)) return true;
    const int64_t cells = (int64_t)d.nx * d.ny, V = (int64_t)d.ny * (d.nx + 1), H = (int64_t)(d.ny + 1) * d.nx;
    const double* area = d.geom + (d.geom_kind == PHX_GEOM_CARTESIAN ? 8 + 11 * ((int64_t)d.nx + d.ny) : 7 * (V + H));
    for (int64_t i = 0; i < cells; ++i)
        if (!(area[i] >= 0x1p-60)) return true;
    return false;
}
bool odd_gas(double gamma, double gm1) {
    return !(gamma >= 0x1p-20 && gamma <= 0x1p20 && gm1 >= 0x1p-20 && gm1 <= 0x1p20);
}

// Work lists: per block, row ranges of `rows` rows times column strips.  The fused variant uses
// STRIP owned columns per item; the split variant uses STRIP_A for its reconstruction kernel,
// STRIP_B with `rows` face rows (ny + 1 of them) for the y-face kernel and STRIP_B with rows_b rows
// for the update kernel.
void release_graphs(phx_plan* P);

// flat y-face stage: lanes per workgroup (rows_b + 1 waves, as the one-face-per-wave stage) and the
// faces its dynamic LDS may hold (64 KiB)
constexpr int FLAT_MAX_FACES = 2048;
int flat_threads(const phx_plan* P) { return (std::min(std::max(P->rows_b, 1), FLAT_MAX_WAVES - 1) + 1) * WAVE; }

// The fused kernel's work list of one geometry kind, arranged for the XCDs.  Workgroup w runs item
// lo_x + (w >> 3) of XCD x = w & 7, whose items are the contiguous range [n x / 8, n (x + 1) / 8)
// (item_range), so each XCD works through its range in list order.
//  * Pairs of consecutive items (neighbouring column strips, or row ranges, of one block) are dealt
//    to the XCDs in turn, so every XCD gets an even share of every case: cases differ in cost per
//    cell (uniform regions skip divisions, cases that failed are skipped), and contiguous ranges of
//    whole cases left some XCDs with less work than others.  (Dealing whole row chunks, all strips
//    of one row range, was 1 % slower on the 64-case batch; single items the same as pairs.)
//  * Every range is made the same length and its last items are split into two halves of their
//    rows: an XCD then finishes on half-size items, which levels the last round of workgroups.
// `tail` = splits per XCD; the set of cells and the work per cell are unchanged.  (Should a range run
// out of items of two or more rows before reaching the common length, the ranges of item_range
// shift against these groups: every item still runs exactly once.)
void order_for_xcds(std::vector<WorkItem>& L, int tail) {
    const int nb = (int)L.size();
    if (tail <= 0 || nb < 8 * 4) return;
    tail = std::min(tail, nb / 8 / 2);
    std::vector<WorkItem> per[8];
    for (int i = 0, g = 0; i < nb; ++g) {
        const int k = std::min(nb, i + 2);
        per[g % 8].insert(per[g % 8].end(), L.begin() + i, L.begin() + k);
        i = k;
    }
    size_t most = 0;
    for (int x = 0; x < 8; ++x) most = std::max(most, per[x].size());
    const int T = (int)most + tail;  // items per XCD after the splits
    std::vector<WorkItem> out;
    out.reserve((size_t)8 * T);
    for (int x = 0; x < 8; ++x) {
        int need = T - (int)per[x].size();
        std::vector<WorkItem>& head = per[x];
        std::vector<WorkItem> back;
        while (need > 0 && !head.empty()) {
            const WorkItem it = head.back();
            head.pop_back();
            if (it.r1 - it.r0 < 2) {
                back.push_back(it);
                continue;
            }
            const int m = it.r0 + (it.r1 - it.r0) / 2;
            back.push_back(WorkItem{it.block, it.j0, m, it.r1});
            back.push_back(WorkItem{it.block, it.j0, it.r0, m});
            --need;
        }
        out.insert(out.end(), head.begin(), head.end());
        out.insert(out.end(), back.rbegin(), back.rend());
    }
    L.swap(out);
}

// A work list dealt to the XCDs in chunks of `chunk` consecutive items: chunk c goes to XCD c mod 8
// (the next XCD with room once one is full), each XCD keeping the range length item_range gives it,
// so every XCD gets a share of every region of the mesh.  Chosen per workload by the autotuner:
// it pays where the cost per cell varies over the mesh (uniform regions skip divisions), and costs
// L2 reuse of the items' shared halo rows and columns where it does not.
void deal_to_xcds(std::vector<WorkItem>& L, int chunk) {
    const int n = (int)L.size();
    if (chunk <= 0 || n < 8 * chunk) return;
    int lo[8], room[8];
    for (int x = 0; x < 8; ++x) {
        lo[x] = (int)((long)n * x / 8);
        room[x] = (int)((long)n * (x + 1) / 8) - lo[x];
    }
    std::vector<WorkItem> out(L.size());
    int used[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = 0, x = 0; i < n; i += chunk, x = (x + 1) % 8)
        for (int q = i; q < std::min(n, i + chunk); ++q) {
            int t = x;
            while (used[t] >= room[t]) t = (t + 1) % 8;
            out[lo[t] + used[t]++] = L[q];
        }
    L.swap(out);
}

int build_items(phx_plan* P) {
    for (int kind = 0; kind < 2; ++kind) {
        P->items[kind].clear();
        P->items_b[kind].clear();
        P->items_f[kind].clear();
        if (P->ditems[kind]) { (void)hipFree(P->ditems[kind]); P->ditems[kind] = nullptr; }
        if (P->ditems_b[kind]) { (void)hipFree(P->ditems_b[kind]); P->ditems_b[kind] = nullptr; }
        if (P->ditems_f[kind]) { (void)hipFree(P->ditems_f[kind]); P->ditems_f[kind] = nullptr; }
        for (int p = 0; p < 3; ++p) {
            P->items_e[p][kind].clear();
            if (P->ditems_e[p][kind]) { (void)hipFree(P->ditems_e[p][kind]); P->ditems_e[p][kind] = nullptr; }
        }
    }
    for (int p = 0; p < 3; ++p) {
        if (P->ditems_em[p]) { (void)hipFree(P->ditems_em[p]); P->ditems_em[p] = nullptr; }
        P->n_em[p] = P->grid_em[p] = 0;
        if (P->ditems_m[p]) { (void)hipFree(P->ditems_m[p]); P->ditems_m[p] = nullptr; }
        P->n_m[p] = P->grid_m[p] = 0;
    }
    const int rows = P->rows_per_item > 0 ? P->rows_per_item : 32;
    const bool split = P->variant == 1 || P->variant >= 5;
    P->flat_q[0] = P->flat_q[1] = 0;
    const int strip = split ? STRIP_A : STRIP;
    const int item_rows = P->variant == 2 ? wg_rows(rows) : rows;  // shared-halo items: one row per inner wave
    for (int b = 0; b < P->nblocks; ++b) {
        const phx_block_desc& d = P->desc[b];
        const int kind = d.geom_kind == PHX_GEOM_CARTESIAN ? 1 : 0;
        for (int r0 = 0; r0 < d.ny; r0 += item_rows)
            for (int j0 = 0; j0 < d.nx; j0 += strip)
                P->items[kind].push_back({b, j0, r0, std::min(r0 + item_rows, d.ny)});
        if (P->variant == 3) {
            const int nc = d.nx * d.ny, nf = d.ny * (d.nx + 1) + (d.ny + 1) * d.nx;
            for (int e = 0; e < nc; e += EW_RCELLS) P->items_e[0][kind].push_back({b, e, std::min(EW_RCELLS, nc - e), 0});
            for (int e = 0; e < nf; e += EW_WG) P->items_e[1][kind].push_back({b, e, std::min(EW_WG, nf - e), 0});
            for (int e = 0; e < nc; e += EW_WG) P->items_e[2][kind].push_back({b, e, std::min(EW_WG, nc - e), 0});
        }
        if (P->variant == 7 || P->variant == 8)  // row-major reconstruction items: LIN_OWN positions each
            for (int p0 = 0; p0 < d.ny * (d.nx + 1); p0 += LIN_OWN) P->items_f[kind].push_back({b, p0, 0, 0});
        if (P->variant == 8) {
            // flat y-face ranges: workgroups of T lanes, q >= rows_per_item faces per lane and at
            // least 64 cells per range (n = q*T - nx)
            const int T = flat_threads(P), nc = d.nx * d.ny;
            const int qmin = (d.nx + 64 + T - 1) / T;  // phx_set_variant checked qmin * T <= FLAT_MAX_FACES
            const int q = std::min(std::max(P->rows_per_item, qmin), FLAT_MAX_FACES / T);
            P->flat_q[kind] = std::max(P->flat_q[kind], q);
            const int n = q * T - d.nx;
            for (int c0 = 0; c0 < nc; c0 += n) P->items_b[kind].push_back({b, c0, std::min(n, nc - c0), 0});
        }
        if (P->variant == 5 || P->variant == 6 || P->variant == 7) {
            const int rb = P->variant != 5 ? std::min(std::max(P->rows_b, 1), YU_MAX_ROWS) : P->rows_b;
            for (int r0 = 0; r0 < d.ny; r0 += rb)
                for (int j0 = 0; j0 < d.nx; j0 += STRIP_B)
                    P->items_b[kind].push_back({b, j0, r0, std::min(r0 + rb, d.ny)});
        }
        if (P->variant == 1) {
            for (int r0 = 0; r0 <= d.ny; r0 += rows)
                for (int j0 = 0; j0 < d.nx; j0 += STRIP_B)
                    P->items_f[kind].push_back({b, j0, r0, std::min(r0 + rows, d.ny + 1)});
            for (int r0 = 0; r0 < d.ny; r0 += P->rows_b)
                for (int j0 = 0; j0 < d.nx; j0 += STRIP_B)
                    P->items_b[kind].push_back({b, j0, r0, std::min(r0 + P->rows_b, d.ny)});
        }
    }
    // fused kernel, one workgroup per item: item pairs dealt to the XCDs, half a round of
    // workgroups per XCD (3 waves on each of its SIMDs) ending on half-size items, but no more than a sixth
    // of the items, whose halo rows cost more than the even end gives (1.4 x 10^6 cells, 2,400 items: us
    // per stage 116 with 192 per XCD, 114 with 48; batch of 2.4 x 10^6, 196 and 192; 64 cases of 6 x 10^6
    // and 9,800 items the other way, 447 and 464)
    if (P->variant == 0 && P->grid_waves == 0)
        for (int kind = 0; kind < 2; ++kind) order_for_xcds(P->items[kind], std::min(P->ncu * 4 * 3 / 8 / 2, (int)P->items[kind].size() / 8 / 6));
    if (P->variant != 0 && P->grid_waves == 0 && P->xcd_chunk > 0)
        for (int kind = 0; kind < 2; ++kind) {
            deal_to_xcds(P->items[kind], P->xcd_chunk);
            deal_to_xcds(P->items_b[kind], P->xcd_chunk);
            deal_to_xcds(P->items_f[kind], P->xcd_chunk);
            for (int p = 0; p < 3; ++p) deal_to_xcds(P->items_e[p][kind], P->xcd_chunk);
        }
    int rc = upload_items(P, P->items, P->ditems, P->grid, P->grid_waves);
    if (rc) return rc;
    rc = upload_items(P, P->items_b, P->ditems_b, P->grid_b, P->grid_waves);
    if (rc) return rc;
    rc = upload_items(P, P->items_f, P->ditems_f, P->grid_f, P->grid_waves);
    if (rc) return rc;
    for (int p = 0; p < 3; ++p) {
        rc = upload_items(P, P->items_e[p], P->ditems_e[p], P->grid_e[p], P->grid_waves);
        if (rc) return rc;
    }
    // both geometry kinds: one list of the shared-halo stage, and per phase of the element-wise stage and of
    // the split stages 6 and 7 with midpoint faces (one launch instead of two; the kernels choose the path per block)
    auto merge = [&](const std::vector<WorkItem> (&two)[2], DevItem*& dev, int& n_out, int& grid_out) -> int {
        if (two[0].empty() || two[1].empty()) return PHX_OK;
        std::vector<WorkItem> both(two[0]);
        both.insert(both.end(), two[1].begin(), two[1].end());
        if (P->grid_waves == 0) deal_to_xcds(both, P->xcd_chunk);
        const size_t n = both.size();
        const int rc = upload_list(P, both, dev);
        if (rc) return rc;
        n_out = (int)n;
        grid_out = (int)((P->grid_waves > 0 && (size_t)P->grid_waves < n) ? P->grid_waves : n);
        return PHX_OK;
    };
    if (P->variant == 3)
        for (int p = 0; p < 3; ++p) {
            rc = merge(P->items_e[p], P->ditems_em[p], P->n_em[p], P->grid_em[p]);
            if (rc) return rc;
        }
    if (P->variant == 2) {
        rc = merge(P->items, P->ditems_m[0], P->n_m[0], P->grid_m[0]);
        if (rc) return rc;
    }
    if ((P->variant == 6 || P->variant == 7) && P->ph.nq == 1) {
        rc = merge(P->items_b, P->ditems_m[1], P->n_m[1], P->grid_m[1]);
        if (rc) return rc;
        if (P->variant == 6) rc = merge(P->items, P->ditems_m[0], P->n_m[0], P->grid_m[0]);
        else rc = merge(P->items_f, P->ditems_m[2], P->n_m[2], P->grid_m[2]);
        if (rc) return rc;
    }
    release_graphs(P);
    return PHX_OK;
}

// Destroys the captured step graphs (they hold the launch list and the state pointer).
void release_graphs(phx_plan* P) {
    for (int g = 0; g < GRAPHS; ++g) {
        if (P->gexec[g]) { (void)hipGraphExecDestroy(P->gexec[g]); P->gexec[g] = nullptr; }
        if (P->graph[g]) { (void)hipGraphDestroy(P->graph[g]); P->graph[g] = nullptr; }
    }
    P->graph_U = nullptr;
}

StageArgs base_args(phx_plan* P) {
    StageArgs A;
    memset(&A, 0, sizeof(A));
    A.blocks = P->dblocks;
    A.state_out = -1;
    A.dt = P->dt;
    A.bad = P->bad;
    A.nslot = P->nslot;
    A.step = P->step;
    A.ph = P->ph;
    return A;
}

// one launch of kernel family T over the items of one geometry kind; minw = register budget asked for
// (2, 3 or 4)
template <class T>
void launch_kind(const phx_plan* P, StageArgs& S, int kind, const DevItem* items, int nitems, int grid, int minw,
                 hipStream_t st) {
    StageArgs A = S;
    A.items = items;
    A.nitems = nitems;
    T::launch(P, kind, minw, dim3(grid + A.fold_blocks), st, A);
    S.fold_blocks = 0;  // the stage's first launch takes the extra workgroups
}

// One phase of a stage over both geometry kinds: launch(kind, stream) for each kind that has work.
// With work of both kinds, kind 1 runs on the plan's side stream concurrently with kind 0 on st
// (fork and join through events, which a graph capture turns into parallel branches): the kinds
// write disjoint blocks and read only what earlier phases wrote (inter-block outer states are cell
// averages of the stage input), and their per-case CFL and realizability reductions are atomic
// minima, so the order of the two launches does not change any result.  On mixed meshes of a few
// thousand cells the launches, not the arithmetic, set the time of a phase.
template <class F>
void for_kinds(phx_plan* P, bool has0, bool has1, hipStream_t st, F&& launch) {
    if (has0 && has1 && P->side_stream && hipEventRecord(P->ev_fork, st) == hipSuccess &&
        hipStreamWaitEvent(P->side_stream, P->ev_fork, 0) == hipSuccess) {
        launch(1, P->side_stream);
        launch(0, st);
        if (hipEventRecord(P->ev_join, P->side_stream) != hipSuccess ||
            hipStreamWaitEvent(st, P->ev_join, 0) != hipSuccess)
            (void)hipStreamSynchronize(P->side_stream);  // join on the host instead
        return;
    }
    if (has0) launch(0, st);
    if (has1) launch(1, st);
}

void launch_stage(phx_plan* P, StageArgs A, hipStream_t st) {
    if (P->variant == 8) {
        A.sn = P->sn;
        A.p1 = P->p1;
        A.rows_wave = flat_threads(P) / WAVE - 1;
        for_kinds(P, !P->items_f[0].empty(), !P->items_f[1].empty(), st, [&](int kind, hipStream_t s) {
            launch_kind<k_recon_x_lin_tag>(P, A, kind, P->ditems_f[kind], (int)P->items_f[kind].size(),
                                           P->grid_f[kind], P->waves_per_simd, s);
        });
        for_kinds(P, !P->items_b[0].empty(), !P->items_b[1].empty(), st, [&](int kind, hipStream_t s) {
            StageArgs Ak = A;
            Ak.fq = P->flat_q[kind];
            launch_kind<k_yface_update_flat_tag>(P, Ak, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                 P->grid_b[kind], 2, s);
        });
        return;
    }
    if (P->variant == 7) {
        A.sn = P->sn;
        A.p1 = P->p1;
        A.rows_wave = std::min(std::max(P->rows_b, 1), YU_MAX_ROWS);
        if (P->ditems_m[2]) launch_recon_x_lin_mixed(P, A, st);  // (takes A.fold_blocks; the others ignore them)
        else
            for_kinds(P, !P->items_f[0].empty(), !P->items_f[1].empty(), st, [&](int kind, hipStream_t s) {
                launch_kind<k_recon_x_lin_tag>(P, A, kind, P->ditems_f[kind], (int)P->items_f[kind].size(),
                                               P->grid_f[kind], P->waves_per_simd, s);
            });
        if (P->ditems_m[1]) launch_yface_wg_mixed(P, A, st);
        else
            for_kinds(P, !P->items_b[0].empty(), !P->items_b[1].empty(), st, [&](int kind, hipStream_t s) {
                launch_kind<k_yface_update_wg_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                   P->grid_b[kind], 2, s);
            });
        return;
    }
    if (P->variant == 6) {
        A.sn = P->sn;
        A.p1 = P->p1;
        A.rows_wave = std::min(std::max(P->rows_b, 1), YU_MAX_ROWS);
        const bool gauss = P->ph.nq > 1;
        if (!gauss && P->ditems_m[0] && P->ditems_m[1]) {
            launch_recon_x_mixed(P, A, st);
            launch_yface_wg_mixed(P, A, st);
            return;
        }
        for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_recon_x_q_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                             P->grid[kind], 2, s);
            else
                launch_kind<k_recon_x_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                           P->grid[kind], P->waves_per_simd, s);
        });
        for_kinds(P, !P->items_b[0].empty(), !P->items_b[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_yface_update_wg_q_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                     P->grid_b[kind], 2, s);
            else
                launch_kind<k_yface_update_wg_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                   P->grid_b[kind], 2, s);
        });
        return;
    }
    if (P->variant == 5) {
        A.sn = P->sn;
        A.p1 = P->p1;
        const bool gauss = P->ph.nq > 1;
        for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_recon_x_q_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                             P->grid[kind], 2, s);
            else
                launch_kind<k_recon_x_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                           P->grid[kind], P->waves_per_simd, s);
        });
        for_kinds(P, !P->items_b[0].empty(), !P->items_b[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_yface_update_q_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                  P->grid_b[kind], 2, s);
            else
                launch_kind<k_yface_update_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(),
                                                P->grid_b[kind], 2, s);
        });
        return;
    }
    if (P->variant == 1) {
        A.sn = P->sn;
        A.p1 = P->p1;
        const bool gauss = P->ph.nq > 1;
        for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_recon_x_q_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                             P->grid[kind], 2, s);
            else
                launch_kind<k_recon_x_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(),
                                           P->grid[kind], P->waves_per_simd, s);
        });
        A.yf = P->yf;
        for_kinds(P, !P->items_f[0].empty(), !P->items_f[1].empty(), st, [&](int kind, hipStream_t s) {
            if (gauss)
                launch_kind<k_yface_q_tag>(P, A, kind, P->ditems_f[kind], (int)P->items_f[kind].size(),
                                           P->grid_f[kind], 2, s);
            else
                launch_kind<k_yface_tag>(P, A, kind, P->ditems_f[kind], (int)P->items_f[kind].size(),
                                         P->grid_f[kind], 2, s);
        });
        for_kinds(P, !P->items_b[0].empty(), !P->items_b[1].empty(), st, [&](int kind, hipStream_t s) {
            launch_kind<k_update_tag>(P, A, kind, P->ditems_b[kind], (int)P->items_b[kind].size(), P->grid_b[kind],
                                      2, s);
        });
        return;
    }
    if (P->variant == 3) {
        A.rb = P->ew_rb;
        A.ff = P->ew_ff;
        if (P->ditems_em[0]) launch_ew_mixed(P, A, 0, st);
        else
            for_kinds(P, !P->items_e[0][0].empty(), !P->items_e[0][1].empty(), st, [&](int kind, hipStream_t s) {
                launch_kind<k_ew_recon_tag>(P, A, kind, P->ditems_e[0][kind], (int)P->items_e[0][kind].size(),
                                            P->grid_e[0][kind], 2, s);
            });
        if (P->ditems_em[1]) launch_ew_mixed(P, A, 1, st);
        else
            for_kinds(P, !P->items_e[1][0].empty(), !P->items_e[1][1].empty(), st, [&](int kind, hipStream_t s) {
                launch_kind<k_ew_face_tag>(P, A, kind, P->ditems_e[1][kind], (int)P->items_e[1][kind].size(),
                                           P->grid_e[1][kind], 2, s);
            });
        if (P->ditems_em[2]) launch_ew_mixed(P, A, 2, st);
        else
            for_kinds(P, !P->items_e[2][0].empty(), !P->items_e[2][1].empty(), st, [&](int kind, hipStream_t s) {
                launch_kind<k_ew_update_tag>(P, A, kind, P->ditems_e[2][kind], (int)P->items_e[2][kind].size(),
                                             P->grid_e[2][kind], 2, s);
            });
        return;
    }
    if (P->variant == 4) {
        for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
            launch_kind<k_stage_pair_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(), P->grid[kind],
                                          std::min(P->waves_per_simd, 3), s);
        });
        return;
    }
    if (P->variant == 2) {
        A.rows_wave = wg_rows(P->rows_per_item);
        if (P->ditems_m[0]) {
            launch_stage_wg_mixed(P, A, st);
            return;
        }
        for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
            launch_kind<k_stage_wg_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(), P->grid[kind],
                                        2, s);
        });
        return;
    }
    // the fused kernel needs more than 128 registers: at most 3 waves per SIMD
    for_kinds(P, !P->items[0].empty(), !P->items[1].empty(), st, [&](int kind, hipStream_t s) {
        launch_kind<k_stage_tag>(P, A, kind, P->ditems[kind], (int)P->items[kind].size(), P->grid[kind],
                                 std::min(P->waves_per_simd, 3), s);
    });
}

void launch_dt_reduce(phx_plan* P, const double* U, hipStream_t st) {
    const int sets = 2 * P->ncases;  // both sets of the minima
    hipLaunchKernelGGL(k_fill_inf, dim3((sets * P->nslot + 255) / 256), dim3(256), 0, st, sets, P->nslot, P->dtmin);
    for (int kind = 0; kind < 2; ++kind) {
        const int n = (int)P->items[kind].size();
        if (!n) continue;
        DtArgs D{P->ditems[kind], n, (P->variant == 1 || P->variant >= 5) ? STRIP_A : STRIP,
                 U, P->dtmin,
                 P->bad, P->step, P->nslot,
                 P->ph};
        if (kind == 1) hipLaunchKernelGGL(k_dt<true>, dim3(P->grid[kind]), dim3(WAVE), 0, st, D);
        else hipLaunchKernelGGL(k_dt<false>, dim3(P->grid[kind]), dim3(WAVE), 0, st, D);
    }
}

void launch_reset(phx_plan* P, const double* t0, int step0, hipStream_t st) {
    for (int c0 = 0; c0 < P->ncases; c0 += RESET_CASES) {
        StartTimes T{};
        std::copy(t0 + c0, t0 + std::min(c0 + RESET_CASES, P->ncases), T.t);
        const int n = c0 == 0 ? std::max(2 * P->ncases * P->nslot, RESET_CASES) : RESET_CASES;
        hipLaunchKernelGGL(k_reset, dim3((n + 255) / 256), dim3(256), 0, st, P->ncases, P->nslot, c0, T, P->t, P->dtmin,
                           P->bad, P->step, step0);
    }
}

// Buffers of one stage-program launch: the caller's state U (read as U0 / stage-0 input, written by
// the last stage) and the stage-state buffer the stage reads (s_read) or writes (s_write).
struct BufMap {
    double *u_read, *u_write, *s_read, *s_write;
};

double* map_buf(phx_plan* P, const BufMap& M, int id, bool write) {
    if (id == BUF_USER) return write ? M.u_write : M.u_read;
    if (id == BUF_S0 || id == BUF_S1) return write ? M.s_write : M.s_read;
    return P->acc[id - BUF_ACC0];
}

// CFL minima a step reads (set = its parity in the run) or writes (the other set)
unsigned long long* dtmin_set(const phx_plan* P, int set) {
    return P->dtmin + (size_t)(set & 1) * P->ncases * P->nslot * DT_STRIDE;
}

// Whether a step's kernels take the closing of the step before along (StepFold).  The fused and paired
// stages do not: they run meshes whose steps take 100 times as long.
bool folds(const phx_plan* P) {
    return P->variant == 2 ? P->progs.size() > 1 : P->variant != 0 && P->variant != 4;
}

// dt, times and counter of the next step as a kernel, where the step's own kernels do not take it along
void open_step(phx_plan* P, int parity, const double* frozen, hipStream_t st) {
    if (folds(P)) return;
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(FIN_THREADS), 0, st, P->ncases, P->nslot, P->ph.cfl,
                       dtmin_set(P, parity), P->tfinal, P->t, P->dt, P->step, P->bad, frozen, 1);
}

// What stage s of a step takes along; parity as in open_step
void fold_step_into(const phx_plan* P, StageArgs& A, size_t s, int parity, const double* frozen) {
    if (!folds(P) || s > (P->variant == 2 ? 1 : 0)) return;
    A.fold_mode = P->variant != 2 ? FOLD_ALL : (s == 0 ? FOLD_DT : FOLD_TIME);
    A.fold_set = parity & 1;
    A.fold_blocks = (P->ncases * P->nslot + WAVE - 1) / WAVE;
    A.fold = P->fold;
    A.frozen = frozen;
}

// A stage's place in a step: the step's number in the run (its parity counts) and its schedule
struct InStep {
    int number;
    const double* frozen;
};

// step: null for a stage on its own, which takes nothing along
void launch_prog_stage_mapped(phx_plan* P, size_t s, const BufMap& M, hipStream_t st,
                              const InStep* step) {
    const StageProg& g = P->progs[s];
    StageArgs A = base_args(P);
    if (step) fold_step_into(P, A, s, step->number, step->frozen);
    A.Uin = map_buf(P, M, g.in, false);
    A.nout = (int)g.outs.size();
    for (int m = 0; m < A.nout; ++m) {
        A.dst[m] = map_buf(P, M, g.outs[m].dst, true);
        A.src[m] = map_buf(P, M, g.outs[m].src, false);
        A.a[m] = g.outs[m].a;
    }
    A.state_out = g.state_out;
    A.skip_dead = 1;
    if (g.state_out >= 0) A.dtmin = dtmin_set(P, step ? step->number + 1 : 1);
    launch_stage(P, A, st);
}

void launch_prog_stage(phx_plan* P, double* U, size_t s, hipStream_t st,
                       const InStep* step = nullptr) {
    const StageProg& g = P->progs[s];
    int sw = BUF_S0;
    for (const StageOut& o : g.outs)
        if (o.dst == BUF_S0 || o.dst == BUF_S1) sw = o.dst;
    const BufMap M{U, U, buf_ptr(P, U, g.in == BUF_USER ? BUF_S0 : g.in), buf_ptr(P, U, sw)};
    launch_prog_stage_mapped(P, s, M, st, step);
}

// one step, the number-th of its run (from launch_dt_reduce, or with a schedule)
void launch_step(phx_plan* P, double* U, hipStream_t st, const double* frozen, int number) {
    open_step(P, number, frozen, st);
    const InStep step{number, frozen};
    for (size_t s = 0; s < P->progs.size(); ++s) launch_prog_stage(P, U, s, st, &step);
    if (P->copy_back)
        (void)hipMemcpyAsync(U, P->sbuf[0], (size_t)P->state_len * sizeof(double), hipMemcpyDeviceToDevice, st);
}

}  // namespace

extern "C" {

const char* phx_last_error(void) { return g_err.c_str(); }

int64_t phx_state_len(const phx_plan* P) { return P ? P->state_len : -1; }

int phx_plan_destroy(phx_plan* P) {
    if (!P) return PHX_OK;
    (void)hipDeviceSynchronize();
    phx::host::adjoint_release(P);
    release_graphs(P);
    if (P->cap_stream) (void)hipStreamDestroy(P->cap_stream);
    if (P->ev_a) (void)hipEventDestroy(P->ev_a);
    if (P->ev_b) (void)hipEventDestroy(P->ev_b);
    if (P->side_stream) (void)hipStreamDestroy(P->side_stream);
    if (P->ev_fork) (void)hipEventDestroy(P->ev_fork);
    if (P->ev_join) (void)hipEventDestroy(P->ev_join);
    void* ptrs[] = {P->dblocks, P->dgeom, P->ditems[0], P->ditems[1], P->ditems_b[0], P->ditems_b[1], P->ditems_f[0],
                    P->ditems_f[1], P->sn, P->p1, P->yf, P->ew_rb, P->ew_ff, P->ditems_e[0][0], P->ditems_e[0][1],
                    P->ditems_e[1][0], P->ditems_e[1][1], P->ditems_e[2][0], P->ditems_e[2][1],
                    P->ditems_em[0], P->ditems_em[1], P->ditems_em[2], P->ditems_m[0], P->ditems_m[1],
                    P->ditems_m[2],
                    P->sbuf[0], P->sbuf[1], P->t, P->tfinal, P->dtmin, P->fold, P->dghost_off};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    for (int m = 0; m < MAX_ACC; ++m)
        if (P->acc[m]) (void)hipFree(P->acc[m]);
    delete P;
    return PHX_OK;
}

int phx_plan_create(const phx_plan_desc* D, phx_plan** out) {
    if (!D || !out) return fail(PHX_E_INVALID, "null argument");
    *out = nullptr;
    if (D->abi_version != PHX_ABI_VERSION) return fail(PHX_E_INVALID, "ABI version mismatch");
    if (D->nblocks < 1 || !D->blocks) return fail(PHX_E_INVALID, "no blocks");
    if (D->ncases < 1) return fail(PHX_E_INVALID, "ncases must be >= 1");
    if (D->flux != PHX_FLUX_ROE && D->flux != PHX_FLUX_HLLL)
        return fail(PHX_E_INVALID, "Flux function type is not available.");
    if (D->limiter < PHX_LIMITER_VENKATAKRISHNAN || D->limiter > PHX_LIMITER_VAN_LEER)
        return fail(PHX_E_INVALID, "MUSCL: Slope limiter type not specified.");
    if (D->reconstruction != PHX_RECON_CONSERVATIVE && D->reconstruction != PHX_RECON_PRIMITIVE)
        return fail(PHX_E_INVALID, "unknown reconstruction type");
    if (D->quadrature_points < 1 || D->quadrature_points > PHX_MAX_QUADRATURE_POINTS)
        return fail(PHX_E_INVALID, "quadrature_points must be 1, 2 or 3");
    const int nq = D->quadrature_points;
    if (D->nstages < 1 || D->nstages > PHX_MAX_STAGES || !D->butcher_a)
        return fail(PHX_E_INVALID, "invalid Butcher table");
    if (!D->t_final) return fail(PHX_E_INVALID, "t_final is null");
    int64_t total = 0;
    for (int b = 0; b < D->nblocks; ++b) {
        const phx_block_desc& d = D->blocks[b];
        const std::string where = "block " + std::to_string(b) + ": ";
        if (d.nx < 1 || d.ny < 1) return fail(PHX_E_INVALID, where + "nx, ny must be >= 1");
        if (d.case_id < 0 || d.case_id >= D->ncases) return fail(PHX_E_INVALID, where + "case_id out of range");
        if (d.state_offset < 0 || d.state_offset % 4) return fail(PHX_E_INVALID, where + "state_offset must be a non-negative multiple of 4");
        if (!d.geom) return fail(PHX_E_INVALID, where + "geometry is null");
        int64_t glen;
        if (d.geom_kind == PHX_GEOM_CARTESIAN) glen = 8 + 11LL * d.nx + 11LL * d.ny + (int64_t)d.nx * d.ny;
        else if (d.geom_kind == PHX_GEOM_GENERAL) glen = 7LL * d.ny * (d.nx + 1) + 7LL * (d.ny + 1) * d.nx + 5LL * d.ny * d.nx;
        else return fail(PHX_E_INVALID, where + "unknown geometry kind");
        if (nq > 1) glen += 8LL * nq * d.nx * d.ny;  // Gauss-point offsets
        if (d.geom_len != glen) return fail(PHX_E_INVALID, where + "geometry length mismatch");
        for (int s = 0; s < 4; ++s) {
            const int st = d.side_type[s];
            if (st < PHX_SIDE_NEIGHBOR || st > PHX_SIDE_OUTLET) return fail(PHX_E_INVALID, where + "invalid side type");
            if (st == PHX_SIDE_NEIGHBOR) {
                const int n = d.neighbor[s];
                if (n < 0 || n >= D->nblocks) return fail(PHX_E_INVALID, where + "neighbour index out of range");
                const phx_block_desc& o = D->blocks[n];
                if ((s == PHX_E || s == PHX_W) && o.ny != d.ny) return fail(PHX_E_INVALID, where + "E/W neighbour ny mismatch");
                if ((s == PHX_N || s == PHX_S) && o.nx != d.nx) return fail(PHX_E_INVALID, where + "N/S neighbour nx mismatch");
                if (o.case_id != d.case_id) return fail(PHX_E_INVALID, where + "neighbour belongs to another case");
            }
        }
        total = std::max<int64_t>(total, d.state_offset + 4LL * d.nx * d.ny);
    }
    // overlap check
    {
        std::vector<std::pair<int64_t, int64_t>> iv;
        for (int b = 0; b < D->nblocks; ++b)
            iv.push_back({D->blocks[b].state_offset, D->blocks[b].state_offset + 4LL * D->blocks[b].nx * D->blocks[b].ny});
        std::sort(iv.begin(), iv.end());
        for (size_t i = 1; i < iv.size(); ++i)
            if (iv[i].first < iv[i - 1].second) return fail(PHX_E_INVALID, "block state ranges overlap");
    }

    phx_plan* P = new phx_plan();
    auto bail = [&](int rc) { phx_plan_destroy(P); return rc; };
    int rc;
#define PHX_CKP(call)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) return bail(fail(PHX_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_))); \
    } while (0)
    PHX_CKP(hipGetDevice(&P->device));
    PHX_CKP(hipDeviceGetAttribute(&P->ncu, hipDeviceAttributeMultiprocessorCount, P->device));
    P->nblocks = D->nblocks;
    P->ncases = D->ncases;
    P->nslot = dt_slots_for(D->ncases);
    P->flux = D->flux;
    P->ph = Phys{D->gamma, D->gm1, D->one_over_gm1, D->g_over_gm1, D->cfl, D->limiter,
                 D->reconstruction == PHX_RECON_PRIMITIVE ? 1 : 0, nq};
    P->ph.odd_gas = odd_gas(D->gamma, D->gm1) ? 1 : 0;
    P->desc.assign(D->blocks, D->blocks + D->nblocks);
    P->state_len = total;
    P->rows_per_item = D->rows_per_item > 0 ? D->rows_per_item : 32;
    P->grid_waves = D->grid_waves;

    // geometry upload (each block aligned to 4 doubles)
    std::vector<int64_t> goff(D->nblocks);
    int64_t gtot = 0;
    for (int b = 0; b < D->nblocks; ++b) {
        goff[b] = gtot;
        gtot += (D->blocks[b].geom_len + 3) / 4 * 4;
    }
    PHX_CKP(hipMalloc(&P->dgeom, std::max<int64_t>(gtot, 4) * sizeof(double)));
    for (int b = 0; b < D->nblocks; ++b)
        PHX_CKP(hipMemcpy(P->dgeom + goff[b], D->blocks[b].geom, D->blocks[b].geom_len * sizeof(double), hipMemcpyHostToDevice));
    P->hblocks.resize(D->nblocks);
    std::vector<long long> ghost_off(D->nblocks);
    long long gacc = 0;
    for (int b = 0; b < D->nblocks; ++b) {
        const phx_block_desc& d = D->blocks[b];
        DevBlock& h = P->hblocks[b];
        memset(&h, 0, sizeof(h));
        h.nx = d.nx; h.ny = d.ny; h.case_id = d.case_id; h.kind = d.geom_kind;
        for (int s = 0; s < 4; ++s) { h.side[s] = d.side_type[s]; h.nbr[s] = d.neighbor[s]; }
        h.off = d.state_offset;
        h.yoff = P->yf_len;
        P->yf_len += 4LL * (d.ny + 1) * d.nx;
        h.foff = P->nfaces;
        P->nfaces += (long long)d.ny * (d.nx + 1) + (long long)(d.ny + 1) * d.nx;
        h.geom = P->dgeom + goff[b];
        h.qoff = nq > 1 ? h.geom + (d.geom_len - 8LL * nq * d.nx * d.ny) : nullptr;
        if (d.geom_kind == PHX_GEOM_CARTESIAN)
            for (int q = 0; q < 8; ++q) h.wall[q] = d.geom[q];
        h.odd = odd_geometry(d) ? 1 : 0;
        ghost_off[b] = gacc;
        gacc += 4LL * (2 * d.ny + 2 * d.nx);
    }
    PHX_CKP(hipMalloc(&P->dblocks, D->nblocks * sizeof(DevBlock)));
    PHX_CKP(hipMemcpy(P->dblocks, P->hblocks.data(), D->nblocks * sizeof(DevBlock), hipMemcpyHostToDevice));
    PHX_CKP(hipMalloc(&P->dghost_off, D->nblocks * sizeof(long long)));
    PHX_CKP(hipMemcpy(P->dghost_off, ghost_off.data(), D->nblocks * sizeof(long long), hipMemcpyHostToDevice));

    P->nstages = D->nstages;
    P->butcher.assign(D->butcher_a, D->butcher_a + (size_t)D->nstages * D->nstages);
    rc = build_programs(P, D->nstages, D->butcher_a);
    if (rc) return bail(rc);
    rc = build_items(P);
    if (rc) return bail(rc);
    if (nq > 1) {  // Gauss faces run a split stage: one y-face per wave, 3 cell rows per workgroup
        P->rows_b = 3;
        rc = phx_set_variant(P, 6, 0);
        if (rc) return bail(rc);
    }

    const size_t sbytes = (size_t)std::max<int64_t>(total, 4) * sizeof(double);
    PHX_CKP(hipMalloc(&P->sbuf[0], sbytes));
    if (D->nstages > 2) PHX_CKP(hipMalloc(&P->sbuf[1], sbytes));
    for (int m = 0; m < P->nacc; ++m) PHX_CKP(hipMalloc(&P->acc[m], sbytes));
    const size_t cb = (size_t)D->ncases * sizeof(double);
    // t, dt, bad and step in one piece, which phx_status copies at once
    PHX_CKP(hipMalloc(&P->t, 2 * cb + (D->ncases + 1) * sizeof(int)));
    P->dt = P->t + D->ncases;
    P->bad = reinterpret_cast<int*>(P->dt + D->ncases);
    P->step = P->bad + D->ncases;
    PHX_CKP(hipMalloc(&P->tfinal, cb));
    PHX_CKP(hipMalloc(&P->dtmin, (size_t)2 * D->ncases * P->nslot * DT_STRIDE * sizeof(unsigned long long)));
    const StepFold fold{P->ncases, P->ph.cfl, P->dtmin, P->tfinal, P->t, P->dt, P->step};
    PHX_CKP(hipMalloc(&P->fold, sizeof(fold)));
    PHX_CKP(hipMemcpy(P->fold, &fold, sizeof(fold), hipMemcpyHostToDevice));
    PHX_CKP(hipMemcpy(P->tfinal, D->t_final, cb, hipMemcpyHostToDevice));
    PHX_CKP(hipMemset(P->dt, 0, cb));
    launch_reset(P, std::vector<double>(D->ncases, 0.0).data(), 0, nullptr);
    PHX_CKP(hipGetLastError());
    PHX_CKP(hipDeviceSynchronize());
    rc = phx::host::adjoint_prepare(P);
    if (rc) return bail(rc);
    PHX_CKP(hipStreamCreateWithFlags(&P->cap_stream, hipStreamNonBlocking));
    PHX_CKP(hipEventCreateWithFlags(&P->ev_a, hipEventDisableTiming));
    PHX_CKP(hipEventCreateWithFlags(&P->ev_b, hipEventDisableTiming));
    PHX_CKP(hipStreamCreateWithFlags(&P->side_stream, hipStreamNonBlocking));
    PHX_CKP(hipEventCreateWithFlags(&P->ev_fork, hipEventDisableTiming));
    PHX_CKP(hipEventCreateWithFlags(&P->ev_join, hipEventDisableTiming));
#undef PHX_CKP
    *out = P;
    return PHX_OK;
}

int phx_reset(phx_plan* P, const double* t0_host, int32_t step0, void* stream) {
    if (!P || !t0_host) return fail(PHX_E_INVALID, "null argument");
    hipStream_t st = (hipStream_t)stream;
    launch_reset(P, t0_host, step0, st);
    PHX_CK(hipGetLastError());
    PHX_CK(hipStreamSynchronize(st));
    return PHX_OK;
}

int phx_run(phx_plan* P, double* U, int32_t nsteps, int32_t use_graph, void* stream) {
    if (!P || !U) return fail(PHX_E_INVALID, "null argument");
    if (nsteps < 0) return fail(PHX_E_INVALID, "nsteps must be >= 0");
    hipStream_t st = (hipStream_t)stream;
    launch_dt_reduce(P, U, st);
    PHX_CK(hipGetLastError());
    if (!use_graph) {
        for (int s = 0; s < nsteps; ++s) launch_step(P, U, st, nullptr, s);
        PHX_CK(hipGetLastError());
        return PHX_OK;
    }
    if (P->graph_U != U) release_graphs(P);
    // The largest graph while enough steps remain, then one graph for each bit of the rest, largest
    // first: every graph but the last starts after an even number of steps, so that one capture of each
    // size fits the alternation of the minima.  All captured on first use, so that later calls only replay.
    const int most = 1 << (GRAPHS - 1);
    for (int g = 0; g < GRAPHS; ++g) {
        if (P->gexec[g]) continue;
        PHX_CK(hipStreamBeginCapture(P->cap_stream, hipStreamCaptureModeThreadLocal));
        for (int s = 0; s < 1 << g; ++s) launch_step(P, U, P->cap_stream, nullptr, s);
        PHX_CK(hipStreamEndCapture(P->cap_stream, &P->graph[g]));
        PHX_CK(hipGraphInstantiate(&P->gexec[g], P->graph[g], nullptr, nullptr, 0));
    }
    P->graph_U = U;
    PHX_CK(hipEventRecord(P->ev_a, st));
    PHX_CK(hipStreamWaitEvent(P->cap_stream, P->ev_a, 0));
    for (int s = 0; s < nsteps / most; ++s) PHX_CK(hipGraphLaunch(P->gexec[GRAPHS - 1], P->cap_stream));
    for (int g = GRAPHS - 2; g >= 0; --g)
        if ((nsteps >> g) & 1) PHX_CK(hipGraphLaunch(P->gexec[g], P->cap_stream));
    PHX_CK(hipEventRecord(P->ev_b, P->cap_stream));
    PHX_CK(hipStreamWaitEvent(st, P->ev_b, 0));
    return PHX_OK;
}

int phx_run_frozen(phx_plan* P, double* U, int32_t nsteps, const double* dt_sched, void* stream) {
    if (!P || !U || (!dt_sched && nsteps > 0)) return fail(PHX_E_INVALID, "null argument");
    hipStream_t st = (hipStream_t)stream;
    for (int s = 0; s < nsteps; ++s) launch_step(P, U, st, dt_sched + (size_t)s * P->ncases, s);
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_run_record(phx_plan* P, double* U, int32_t nsteps, const double* dt_sched, double* stages, void* stream) {
    if (!P || !U || ((!dt_sched || !stages) && nsteps > 0)) return fail(PHX_E_INVALID, "null argument");
    if (nsteps < 0) return fail(PHX_E_INVALID, "nsteps must be >= 0");
    hipStream_t st = (hipStream_t)stream;
    const size_t len = (size_t)P->state_len;
    const int S = (int)P->progs.size();
    if (nsteps == 0) return PHX_OK;
    // The records are the working buffers: step n reads its input from record (n, 0), writes the
    // state of stage s+1 into record (n, s+1) and its result into record (n+1, 0) (U after the last
    // step), so only the first input is copied.
    PHX_CK(hipMemcpyAsync(stages, U, len * sizeof(double), hipMemcpyDeviceToDevice, st));
    for (int n = 0; n < nsteps; ++n) {
        const double* frozen = dt_sched + (size_t)n * P->ncases;
        open_step(P, n, frozen, st);
        const InStep step{n, frozen};
        double* rec = stages + (size_t)n * S * len;
        double* next = (n + 1 < nsteps) ? rec + (size_t)S * len : U;
        for (int s = 0; s < S; ++s) {
            BufMap M;
            M.u_read = rec;
            M.u_write = next;
            M.s_read = rec + (size_t)s * len;
            M.s_write = (s + 1 < S) ? rec + (size_t)(s + 1) * len : next;  // one-stage tables write S0
            launch_prog_stage_mapped(P, (size_t)s, M, st, &step);
        }
    }
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_stage(phx_plan* P, double* U, int32_t stage, void* stream) {
    if (!P || !U) return fail(PHX_E_INVALID, "null argument");
    if (stage < 0 || stage >= (int)P->progs.size()) return fail(PHX_E_INVALID, "stage index out of range");
    launch_prog_stage(P, U, (size_t)stage, (hipStream_t)stream);
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_residual(phx_plan* P, const double* U, double* R, void* stream) {
    if (!P || !U || !R) return fail(PHX_E_INVALID, "null argument");
    StageArgs A = base_args(P);
    A.Uin = U;
    A.Rout = R;
    A.nout = 0;
    launch_stage(P, A, (hipStream_t)stream);
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_dt(phx_plan* P, const double* U, double* dt_dev, void* stream) {
    if (!P || !U || !dt_dev) return fail(PHX_E_INVALID, "null argument");
    hipStream_t st = (hipStream_t)stream;
    launch_dt_reduce(P, U, st);
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(FIN_THREADS), 0, st, P->ncases, P->nslot, P->ph.cfl, P->dtmin, P->tfinal, P->t,
                       dt_dev, P->step, P->bad, (const double*)nullptr, 0);
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_ghosts(phx_plan* P, const double* U, double* G, void* stream) {
    if (!P || !U || !G) return fail(PHX_E_INVALID, "null argument");
    hipLaunchKernelGGL(k_ghosts, dim3(P->nblocks), dim3(256), 0, (hipStream_t)stream, P->dblocks, P->nblocks,
                       P->dghost_off, U, G);
    PHX_CK(hipGetLastError());
    return PHX_OK;
}

int phx_status(phx_plan* P, int32_t* bad_step, int32_t* step, double* t_host, double* dt_host) {
    if (!P) return fail(PHX_E_INVALID, "null argument");
    PHX_CK(hipDeviceSynchronize());
    const size_t n = (size_t)P->ncases;
    std::vector<char> all(2 * n * sizeof(double) + (n + 1) * sizeof(int));
    PHX_CK(hipMemcpy(all.data(), P->t, all.size(), hipMemcpyDeviceToHost));
    const double* t = reinterpret_cast<const double*>(all.data());
    const int* b = reinterpret_cast<const int*>(t + 2 * n);
    if (bad_step)
        for (size_t c = 0; c < n; ++c) bad_step[c] = (b[c] == NEVER) ? -1 : b[c];
    if (step) *step = b[n];
    if (t_host) std::copy(t, t + n, t_host);
    if (dt_host) std::copy(t + n, t + 2 * n, dt_host);
    return PHX_OK;
}

int phx_set_launch(phx_plan* P, int32_t rows_per_item, int32_t grid_waves, int32_t waves_per_simd) {
    if (!P || rows_per_item < 1 || grid_waves < 0 || waves_per_simd < 0 || waves_per_simd > 4 || waves_per_simd == 1)
        return fail(PHX_E_INVALID, "invalid launch parameters");
    PHX_CK(hipDeviceSynchronize());
    P->rows_per_item = rows_per_item;
    P->grid_waves = grid_waves;
    P->waves_per_simd = waves_per_simd == 0 ? 2 : waves_per_simd;
    return build_items(P);
}

int phx_set_variant(phx_plan* P, int32_t variant, int32_t rows_b) {
    if (!P || variant < 0 || variant > 8 || rows_b < 0) return fail(PHX_E_INVALID, "invalid stage variant");
    if (P->ph.nq > 1 && variant != 1 && variant != 5 && variant != 6)
        return fail(PHX_E_INVALID, "more than one Gauss point per face runs the split stages only (variants 1, 5, 6)");
    if (variant == 8) {
        const int rb = rows_b > 0 ? rows_b : P->rows_b;
        const int T = (std::min(std::max(rb, 1), FLAT_MAX_WAVES - 1) + 1) * WAVE;
        for (int b = 0; b < P->nblocks; ++b)
            if ((P->desc[b].nx + 64 + T - 1) / T * T > FLAT_MAX_FACES)
                return fail(PHX_E_INVALID, "a block is too wide for the flat y-face stage (variant 8: nx + 64 faces per range)");
    }
    PHX_CK(hipDeviceSynchronize());
    if ((variant == 1 || variant >= 5) && !P->sn) {
        const size_t L = (size_t)std::max<int64_t>(P->state_len, 4);
        PHX_CK(hipMalloc(&P->sn, 2 * (size_t)std::max(P->ph.nq, 1) * L * sizeof(double)));
        PHX_CK(hipMalloc(&P->p1, L * sizeof(double)));
        PHX_CK(hipMalloc(&P->yf, (size_t)std::max<long long>(P->yf_len, 4) * sizeof(double)));
    }
    if (variant == 3 && !P->ew_rb) {
        const size_t cells = (size_t)std::max<int64_t>(P->state_len, 4) / 4;
        PHX_CK(hipMalloc(&P->ew_rb, phx::adj::RB * cells * sizeof(double)));
        PHX_CK(hipMalloc(&P->ew_ff, 4 * (size_t)std::max<long long>(P->nfaces, 1) * sizeof(double)));
    }
    P->variant = variant;
    if (rows_b > 0) P->rows_b = rows_b;
    return build_items(P);
}

int phx_set_xcd_order(phx_plan* P, int32_t chunk) {
    if (!P || chunk < 0) return fail(PHX_E_INVALID, "invalid XCD chunk (0 or a positive number of work items)");
    PHX_CK(hipDeviceSynchronize());
    P->xcd_chunk = chunk;
    return build_items(P);
}

int phx_launch_info(const phx_plan* P, int32_t* items_cart, int32_t* items_gen, int32_t* grid_cart, int32_t* grid_gen) {
    if (!P) return fail(PHX_E_INVALID, "null argument");
    if (items_cart) *items_cart = (int32_t)P->items[1].size();
    if (items_gen) *items_gen = (int32_t)P->items[0].size();
    if (grid_cart) *grid_cart = P->grid[1];
    if (grid_gen) *grid_gen = P->grid[0];
    return PHX_OK;
}

}  // extern "C"
