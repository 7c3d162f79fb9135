// phx_stage_recon.hip -- instances and launchers of the split stage's strip reconstruction.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
// Register budget of the strip reconstruction in waves per SIMD for a requested one: its geometry is loaded
// before the arithmetic, which takes about 180 registers; the meshes it is used for have one or two
// waves per SIMD.
constexpr int recon_waves(int requested) { return requested >= 4 ? 3 : 2; }

struct k_recon_x_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        constexpr int MM = recon_waves(G ? 3 : M);
        hipLaunchKernelGGL((k_recon_x<C ? 1 : 0, F, MM, G>), g, dim3(WAVE), 0, st, A);
    }
};
}  // namespace

void k_recon_x_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_recon_x_go>(P, kind, minw, g, st, A);
}

// one launch of the reconstruction kernel of variant 6 over the merged list of both geometry kinds
void launch_recon_x_mixed(const phx_plan* P, StageArgs A, hipStream_t st) {
    A.items = P->ditems_m[0];
    A.nitems = P->n_m[0];
    const dim3 g(P->grid_m[0] + A.fold_blocks), b(WAVE);
    const bool gen = generic_instance(P), roe = P->flux == PHX_FLUX_ROE;
    const bool w4 = !gen && P->waves_per_simd >= 4;  // recon_waves: the budgets of the launches per kind
#define PHX_RX(F, M, G) hipLaunchKernelGGL((k_recon_x<2, F, M, G>), g, b, 0, st, A)
    if (gen) { if (roe) PHX_RX(0, 2, true); else PHX_RX(1, 2, true); }
    else if (w4) { if (roe) PHX_RX(0, 3, false); else PHX_RX(1, 3, false); }
    else { if (roe) PHX_RX(0, 2, false); else PHX_RX(1, 2, false); }
#undef PHX_RX
}

}  // namespace stage
}  // namespace phx
