// k_systolic_tile for MXQUANT's ladders.
#include "systolic_tile_impl.h"

void mxq_sys::launch_tile_mxquant(int kind, dim3 grid, const SysArgs& a, const FastLanes& fl, hipStream_t st) {
  if (kind == kMxqFinal) launch_tile_ladder<kMxqFinal, 16, true>(grid, a, fl, st);
  else if (kind == kMxq) launch_tile_size<kMxq, false>(grid, a, fl, st);
  else launch_tile_size<kMxqHigh, false>(grid, a, fl, st);
}
