#include "norm_linear_impl.hpp"

namespace clusten {

int launch_norm_linear_f16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_F16) return launch_norm_linear_typed<f16_t, f16_t>(a, C, stream);
    return launch_norm_linear_typed<f16_t, float>(a, C, stream);
}

}  // namespace clusten
