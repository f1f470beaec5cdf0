// k_mlp_backward_shared instantiations: bf16_t weights, None and LeakyReLU.
#include "mlp_bwd_shared.hpp"

namespace nect {

int32_t launch_mlp_backward_shared_bf16_pwl(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    return launch_mlp_backward_shared<bf16_t, false, 1, 7>(a, workgroups, st);
}

}  // namespace nect
