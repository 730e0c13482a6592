// k_systolic_small for MXQUANT's ladders.
#include "systolic_small_impl.h"

void mxq_sys::launch_small_mxquant(int kind, const SysArgs& a, const FastLanes& fl, const SmallTile& t, int64_t count,
                                   hipStream_t st) {
  if (kind == kMxqFinal) launch_small_ladder<kMxqFinal, 16, true>(a, fl, t, count, st);
  else if (kind == kMxq) launch_small_size<kMxq, false>(a, fl, t, count, st);
  else launch_small_size<kMxqHigh, false>(a, fl, t, count, st);
}
