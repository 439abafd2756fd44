// The slice kernel (slice.hpp) for fp16 data, fp16 sums.
#include "slice.hpp"

namespace remifa {
int slice_f16h_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid) {
  return rl ? launch_ib<half_t, SM_F16_H, true>(h, ib, g, grid)
            : launch_ib<half_t, SM_F16_H, false>(h, ib, g, grid);
}
}  // namespace remifa
