#include "block_tail_impl.hpp"

namespace clusten {

int launch_block_tail_bf16(const BlockTailArgs& a, int x_dtype, int C, hipStream_t stream) {
    if (x_dtype == CLUSTEN_BF16) return launch_block_tail_typed<bf16_t, bf16_t>(a, C, stream);
    return launch_block_tail_typed<bf16_t, float>(a, C, stream);
}

}  // namespace clusten
