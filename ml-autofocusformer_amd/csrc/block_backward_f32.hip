#include "block_backward_impl.hpp"

namespace clusten {

int launch_block_tail_backward_f32(const BlockTailGrad& a, int C, hipStream_t stream) { return launch_backward_typed<float, float>(a, C, stream); }
int launch_norm_linear_backward_f32(const NormLinearGrad& a, int C, hipStream_t stream) { return launch_backward_typed<float, float>(a, C, stream); }

}  // namespace clusten
