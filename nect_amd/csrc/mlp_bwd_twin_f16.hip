// k_mlp_backward_twin instantiations: _Float16 weights, 1-4 hidden layers, inputs of up to 64 features.
#include "mlp_bwd_twin.hpp"

namespace nect {

int32_t launch_mlp_backward_twin_f16(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    return launch_mlp_backward_twin<_Float16, 1, 4>(a, workgroups, st);
}

}  // namespace nect
