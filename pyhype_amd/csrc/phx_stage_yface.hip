// phx_stage_yface.hip -- instances and launchers of the split stage's y-face and update kernels
// and of the Gauss-face kernels.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
struct k_yface_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface<C, F, G>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_yface_update_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface_update<C, F, G>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_yface_update_wg_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface_update_wg<C ? 1 : 0, F, G, false>), g, dim3((A.rows_wave + 1) * WAVE), 0, st, A);
    }
};
struct k_yface_update_flat_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        const int T = (A.rows_wave + 1) * WAVE;
        hipLaunchKernelGGL((k_yface_update_flat<C, F, G>), g, dim3(T), (size_t)A.fq * T * sizeof(Q4), st, A);
    }
};
struct k_update_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_update<C>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_recon_x_q_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_recon_x_q<C, F>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_yface_q_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface_q<C, F>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_yface_update_q_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface_update_q<C, F>), g, dim3(WAVE), 0, st, A);
    }
};
struct k_yface_update_wg_q_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        hipLaunchKernelGGL((k_yface_update_wg<C ? 1 : 0, F, true, true>), g, dim3((A.rows_wave + 1) * WAVE), 0, st, A);
    }
};
}  // namespace

void k_recon_x_q_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_recon_x_q_go>(P, kind, minw, g, st, A);
}
void k_yface_q_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_q_go>(P, kind, minw, g, st, A);
}
void k_yface_update_q_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_update_q_go>(P, kind, minw, g, st, A);
}
void k_yface_update_wg_q_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_update_wg_q_go>(P, kind, minw, g, st, A);
}
void k_yface_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_go>(P, kind, minw, g, st, A);
}
void k_yface_update_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_update_go>(P, kind, minw, g, st, A);
}
void k_yface_update_wg_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_update_wg_go>(P, kind, minw, g, st, A);
}
void k_yface_update_flat_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_yface_update_flat_go>(P, kind, minw, g, st, A);
}
void k_update_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_update_go>(P, kind, minw, g, st, A);
}

void launch_yface_wg_mixed(const phx_plan* P, StageArgs A, hipStream_t st) {
    A.items = P->ditems_m[1];
    A.nitems = P->n_m[1];
    const dim3 g(P->grid_m[1]), b((A.rows_wave + 1) * WAVE);
    const bool gen = generic_instance(P), roe = P->flux == PHX_FLUX_ROE;
    if (roe && gen) hipLaunchKernelGGL((k_yface_update_wg<2, 0, true, false>), g, b, 0, st, A);
    else if (roe) hipLaunchKernelGGL((k_yface_update_wg<2, 0, false, false>), g, b, 0, st, A);
    else if (gen) hipLaunchKernelGGL((k_yface_update_wg<2, 1, true, false>), g, b, 0, st, A);
    else hipLaunchKernelGGL((k_yface_update_wg<2, 1, false, false>), g, b, 0, st, A);
}

}  // namespace stage
}  // namespace phx
