// k_systolic_tile for MXGEMMINI's ladders of e4 lanes.
#include "systolic_tile_impl.h"

void mxq_sys::launch_tile_e4(int kind, bool bf16_last, dim3 grid, const SysArgs& a, const FastLanes& fl,
                               hipStream_t st) {
  if (kind == kE4Final) launch_tile_ladder<kE4Final, 16, true>(grid, a, fl, st);
  else if (bf16_last) launch_tile_size<kE4, true>(grid, a, fl, st);
  else launch_tile_size<kE4, false>(grid, a, fl, st);
}
