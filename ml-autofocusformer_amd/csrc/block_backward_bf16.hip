#include "block_backward_impl.hpp"

namespace clusten {

int launch_block_tail_backward_bf16(const BlockTailGrad& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_BF16) return launch_backward_typed<bf16_t, bf16_t>(a, C, stream);
    return launch_backward_typed<bf16_t, float>(a, C, stream);
}
int launch_norm_linear_backward_bf16(const NormLinearGrad& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_BF16) return launch_backward_typed<bf16_t, bf16_t>(a, C, stream);
    return launch_backward_typed<bf16_t, float>(a, C, stream);
}

}  // namespace clusten
