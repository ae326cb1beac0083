#include "norm_linear_impl.hpp"

namespace clusten {

int launch_norm_linear_f32(const NormLinearArgs& a, int C, hipStream_t stream) { return launch_norm_linear_typed<float, float>(a, C, stream); }

}  // namespace clusten
