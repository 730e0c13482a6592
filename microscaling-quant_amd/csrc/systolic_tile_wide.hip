// k_systolic_tile for MXGEMMINI's ladders of wide lanes.
#include "systolic_tile_impl.h"

void mxq_sys::launch_tile_wide(dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st) {
  launch_tile_size<kWide, false>(grid, a, fl, st);
}
