// The slice kernel (slice.hpp) for fp32 data, fp32 sums.
#include "slice.hpp"

namespace remifa {
int slice_f32_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid) {
  return rl ? launch_ib<float, SM_F32, true>(h, ib, g, grid)
            : launch_ib<float, SM_F32, false>(h, ib, g, grid);
}
}  // namespace remifa
