// The slice kernel (slice.hpp) for fp16 data, fp16 operands, fp32 sums.
#include "slice.hpp"

namespace remifa {
int slice_f16tc_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid) {
  return rl ? launch_ib<half_t, SM_F16_TC, true>(h, ib, g, grid)
            : launch_ib<half_t, SM_F16_TC, false>(h, ib, g, grid);
}
}  // namespace remifa
