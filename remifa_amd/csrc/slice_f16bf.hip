// The slice kernel (slice.hpp) for fp16 data, bf16 operands.
#include "slice.hpp"

namespace remifa {
int slice_f16bf_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid) {
  return rl ? launch_ib<half_t, SM_F16_BF, true>(h, ib, g, grid)
            : launch_ib<half_t, SM_F16_BF, false>(h, ib, g, grid);
}
}  // namespace remifa
