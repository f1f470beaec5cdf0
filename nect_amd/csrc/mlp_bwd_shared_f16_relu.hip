// k_mlp_backward_shared instantiations: _Float16 weights, ReLU.
#include "mlp_bwd_shared.hpp"

namespace nect {

int32_t launch_mlp_backward_shared_f16_pwl(const MlpArgs &a, unsigned workgroups, hipStream_t st);

int32_t launch_mlp_backward_shared_f16(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    if (a.d.activation != NECT_ACT_RELU) return launch_mlp_backward_shared_f16_pwl(a, workgroups, st);
    return launch_mlp_backward_shared<_Float16, true, 1, 7>(a, workgroups, st);
}

}  // namespace nect
