// k_systolic_small for MXGEMMINI's ladders of wide lanes.
#include "systolic_small_impl.h"

void mxq_sys::launch_small_wide(const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count,
                                hipStream_t st) {
  launch_small_size<kWide, false>(a, fl, t, count, st);
}
