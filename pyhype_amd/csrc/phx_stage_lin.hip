// phx_stage_lin.hip -- instances and launchers of the split stage's row-major reconstruction.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
struct k_recon_x_lin_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        // HLLL: 128 registers (4 waves per SIMD; 198.4 -> 195.4 us per step of 5 x 500^2 cells), Roe at
        // least 134 (3 waves; 118.3 against 119.9 us on 8 x 150^2 cells)
        constexpr int MM = G ? 3 : (F == 1 || M > 3 ? 4 : 3);
        hipLaunchKernelGGL((k_recon_x_lin<C ? 1 : 0, F, MM, G>), g, dim3(WAVE), 0, st, A);
    }
};
}  // namespace

void k_recon_x_lin_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_recon_x_lin_go>(P, kind, minw, g, st, A);
}

// One launch of the reconstruction kernel of variant 7 over the merged list of both geometry kinds.  Its
// instances hold both kinds' paths: at 4 waves per SIMD the HLLL one spills 57 registers (6 in the
// instances of one kind), so it takes 3 where those take 4 (ramps, us per stage at 3 and 4 waves:
// 4 x 200^2 cells 38.5 and 40.5, 4 x 300^2 57.5 and 60.4, 5 x 500^2 168.9 and 189.7).
void launch_recon_x_lin_mixed(const phx_plan* P, StageArgs A, hipStream_t st) {
    A.items = P->ditems_m[2];
    A.nitems = P->n_m[2];
    const dim3 g(P->grid_m[2] + A.fold_blocks), b(WAVE);
    const bool gen = generic_instance(P), roe = P->flux == PHX_FLUX_ROE;
    const bool w4 = !gen && P->waves_per_simd >= 4;
#define PHX_RX(F, M, G) hipLaunchKernelGGL((k_recon_x_lin<2, F, M, G>), g, b, 0, st, A)
    if (gen) { if (roe) PHX_RX(0, 3, true); else PHX_RX(1, 3, true); }
    else if (w4) { if (roe) PHX_RX(0, 4, false); else PHX_RX(1, 4, false); }
    else { if (roe) PHX_RX(0, 3, false); else PHX_RX(1, 3, false); }
#undef PHX_RX
}

}  // namespace stage
}  // namespace phx
