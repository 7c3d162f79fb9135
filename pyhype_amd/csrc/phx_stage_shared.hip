// phx_stage_shared.hip -- instances and launchers of the shared-halo, paired and element-wise stage kernels.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
struct k_stage_wg_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        constexpr int K = C ? 1 : 0;
        if (A.rows_wave == 1) hipLaunchKernelGGL((k_stage_wg<K, F, 1, G>), g, dim3(wg_waves(1) * WAVE), 0, st, A);
        else hipLaunchKernelGGL((k_stage_wg<K, F, 2, G>), g, dim3(wg_waves(2) * WAVE), 0, st, A);
    }
};
struct k_stage_pair_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        constexpr int MM = G ? 2 : (M > 3 ? 3 : (M < 2 ? 2 : M));
        hipLaunchKernelGGL((k_stage_pair<C, F, MM, G>), g, dim3(PAIR_WAVES * WAVE), 0, st, A);
    }
};
struct k_ew_recon_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_ew_recon<C ? 1 : 0, G>), g, dim3(EW_WG), 0, st, A);
    }
};
struct k_ew_face_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_ew_face<C ? 1 : 0, F, G>), g, dim3(EW_WG), 0, st, A);
    }
};
struct k_ew_update_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_ew_update<C ? 1 : 0>), g, dim3(EW_WG), 0, st, A);
    }
};
}  // namespace

void k_stage_wg_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_stage_wg_go>(P, kind, minw, g, st, A);
}
// one launch over the merged list of both geometry kinds
template <int F, bool G>
static void launch_wg_both(dim3 g, hipStream_t st, const StageArgs& A) {
    if (A.rows_wave == 1) hipLaunchKernelGGL((k_stage_wg<2, F, 1, G>), g, dim3(wg_waves(1) * WAVE), 0, st, A);
    else hipLaunchKernelGGL((k_stage_wg<2, F, 2, G>), g, dim3(wg_waves(2) * WAVE), 0, st, A);
}
void launch_stage_wg_mixed(const phx_plan* P, StageArgs A, hipStream_t st) {
    A.items = P->ditems_m[0];
    A.nitems = P->n_m[0];
    const dim3 g(P->grid_m[0] + A.fold_blocks);
    const bool gen = generic_instance(P);
    if (P->flux == PHX_FLUX_ROE) gen ? launch_wg_both<0, true>(g, st, A) : launch_wg_both<0, false>(g, st, A);
    else gen ? launch_wg_both<1, true>(g, st, A) : launch_wg_both<1, false>(g, st, A);
}
void k_stage_pair_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_stage_pair_go>(P, kind, minw, g, st, A);
}
void k_ew_recon_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_ew_recon_go>(P, kind, minw, g, st, A);
}
void k_ew_face_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_ew_face_go>(P, kind, minw, g, st, A);
}
void k_ew_update_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_ew_update_go>(P, kind, minw, g, st, A);
}

void launch_ew_mixed(const phx_plan* P, StageArgs A, int p, hipStream_t st) {
    A.items = P->ditems_em[p];
    A.nitems = P->n_em[p];
    const dim3 g(P->grid_em[p] + (p == 0 ? A.fold_blocks : 0)), b(EW_WG);
    const bool gen = generic_instance(P), roe = P->flux == PHX_FLUX_ROE;
    if (p == 0) {
        if (gen) hipLaunchKernelGGL((k_ew_recon<2, true>), g, b, 0, st, A);
        else hipLaunchKernelGGL((k_ew_recon<2, false>), g, b, 0, st, A);
    } else if (p == 1) {
        if (roe && gen) hipLaunchKernelGGL((k_ew_face<2, 0, true>), g, b, 0, st, A);
        else if (roe) hipLaunchKernelGGL((k_ew_face<2, 0, false>), g, b, 0, st, A);
        else if (gen) hipLaunchKernelGGL((k_ew_face<2, 1, true>), g, b, 0, st, A);
        else hipLaunchKernelGGL((k_ew_face<2, 1, false>), g, b, 0, st, A);
    } else {
        hipLaunchKernelGGL((k_ew_update<2>), g, b, 0, st, A);
    }
}

}  // namespace stage
}  // namespace phx
