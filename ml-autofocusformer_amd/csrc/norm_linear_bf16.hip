#include "norm_linear_impl.hpp"

namespace clusten {

int launch_norm_linear_bf16(const NormLinearArgs& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_BF16) return launch_norm_linear_typed<bf16_t, bf16_t>(a, C, stream);
    return launch_norm_linear_typed<bf16_t, float>(a, C, stream);
}

}  // namespace clusten
