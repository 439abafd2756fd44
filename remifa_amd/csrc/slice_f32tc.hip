// The slice kernel (slice.hpp) for fp32 data, fp16 operands.
#include "slice.hpp"

namespace remifa {
int slice_f32tc_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid) {
  return rl ? launch_ib<float, SM_F32_TC, true>(h, ib, g, grid)
            : launch_ib<float, SM_F32_TC, false>(h, ib, g, grid);
}
}  // namespace remifa
