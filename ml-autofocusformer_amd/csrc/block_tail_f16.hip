#include "block_tail_impl.hpp"

namespace clusten {

int launch_block_tail_f16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_F16) return launch_block_tail_typed<f16_t, f16_t>(a, C, stream);
    return launch_block_tail_typed<f16_t, float>(a, C, stream);
}

}  // namespace clusten
