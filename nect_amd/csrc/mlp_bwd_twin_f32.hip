// k_mlp_backward_twin instantiations: float weights, 1-3 hidden layers, inputs of up to 64 features.
#include "mlp_bwd_twin.hpp"

namespace nect {

int32_t launch_mlp_backward_twin_f32(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    return launch_mlp_backward_twin<float, 1, 3>(a, workgroups, st);
}

}  // namespace nect
