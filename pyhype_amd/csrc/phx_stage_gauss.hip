// phx_stage_gauss.hip -- instances and launchers of the Gauss-face stage kernels.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
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

}  // namespace stage
}  // namespace phx
