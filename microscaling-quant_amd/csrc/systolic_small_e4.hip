// k_systolic_small for MXGEMMINI's ladders of e4 lanes.
#include "systolic_small_impl.h"

void mxq_sys::launch_small_e4(int kind, bool bf16_last, const SysArgs& a, const FastLanes& fl, const SmallTile& t,
                              int64_t count, hipStream_t st) {
  if (kind == kE4Final) launch_small_ladder<kE4Final, 16, true>(a, fl, t, count, st);
  else if (bf16_last) launch_small_size<kE4, true>(a, fl, t, count, st);
  else launch_small_size<kE4, false>(a, fl, t, count, st);
}
