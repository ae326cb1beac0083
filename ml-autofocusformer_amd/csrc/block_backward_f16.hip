#include "block_backward_impl.hpp"

namespace clusten {

int launch_block_tail_backward_f16(const BlockTailGrad& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_F16) return launch_backward_typed<f16_t, f16_t>(a, C, stream);
    return launch_backward_typed<f16_t, float>(a, C, stream);
}
int launch_norm_linear_backward_f16(const NormLinearGrad& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_F16) return launch_backward_typed<f16_t, f16_t>(a, C, stream);
    return launch_backward_typed<f16_t, float>(a, C, stream);
}

}  // namespace clusten
