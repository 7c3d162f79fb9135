// phx_stage_fused.hip -- instances and launchers of the fused stage kernel.
#include "phx_stage.hpp"

namespace phx {
namespace stage {

namespace {
struct k_stage_go {
    template <bool C, int F, int M, bool G>
    static void go(dim3 g, hipStream_t st, const StageArgs& A) {
        constexpr int MM = G ? 2 : (M > 3 ? 3 : M);
        hipLaunchKernelGGL((k_stage<C, F, MM, G>), g, dim3(WAVE), 0, st, A);
    }
};
}  // namespace

void k_stage_tag::launch(const phx_plan* P, int kind, int minw, dim3 g, hipStream_t st, const StageArgs& A) {
    dispatch<k_stage_go>(P, kind, minw, g, st, A);
}

}  // namespace stage
}  // namespace phx
