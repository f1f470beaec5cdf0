// k_mlp_backward_shared instantiations: _Float16 weights, None and LeakyReLU.
#include "mlp_bwd_shared.hpp"

namespace nect {

int32_t launch_mlp_backward_shared_f16_pwl(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    return launch_mlp_backward_shared<_Float16, false, 1, 7>(a, workgroups, st);
}

}  // namespace nect
