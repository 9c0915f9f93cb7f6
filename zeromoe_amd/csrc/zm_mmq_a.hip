// zm_mmq_a.hip -- instantiations of the grouped int8-MFMA kernel (zm_mmq.hpp) for Q2_K and Q3_K.
#include "zm_mmq.hpp"

namespace zm {

bool mmq_launch_a(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st) {
  if (type == T_Q2_K) return mmq_launch<T_Q2_K>(gateup, tt, nw, items, a, st), true;
  if (type == T_Q3_K) return mmq_launch<T_Q3_K>(gateup, tt, nw, items, a, st), true;
  return false;
}

}  // namespace zm
