// zm_mmq_d.hip -- instantiations of the grouped int8-MFMA kernel (zm_mmq.hpp) for IQ2_XXS and IQ3_XXS.
#include "zm_mmq.hpp"

namespace zm {

bool mmq_launch_d(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st) {
  if (type == T_IQ2_XXS) return mmq_launch<T_IQ2_XXS>(gateup, tt, nw, items, a, st), true;
  if (type == T_IQ3_XXS) return mmq_launch<T_IQ3_XXS>(gateup, tt, nw, items, a, st), true;
  return false;
}

}  // namespace zm
