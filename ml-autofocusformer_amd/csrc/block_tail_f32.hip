#include "block_tail_impl.hpp"

namespace clusten {

int launch_block_tail_f32(const BlockTailArgs& a, int C, hipStream_t stream) { return launch_block_tail_typed<float, float>(a, C, stream); }

}  // namespace clusten
