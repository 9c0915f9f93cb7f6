// zm_mmq_c.hip -- instantiations of the grouped int8-MFMA kernel (zm_mmq.hpp) for Q6_K and IQ4_XS.
#include "zm_mmq.hpp"

namespace zm {

bool mmq_launch_c(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st) {
  if (type == T_Q6_K) return mmq_launch<T_Q6_K>(gateup, tt, nw, items, a, st), true;
  if (type == T_IQ4_XS) return mmq_launch<T_IQ4_XS>(gateup, tt, nw, items, a, st), true;
  return false;
}

}  // namespace zm
