// zm_mmq_b.hip -- instantiations of the grouped int8-MFMA kernel (zm_mmq.hpp) for Q4_K and Q5_K.
#include "zm_mmq.hpp"

namespace zm {

bool mmq_launch_b(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st) {
  if (type == T_Q4_K) return mmq_launch<T_Q4_K>(gateup, tt, nw, items, a, st), true;
  if (type == T_Q5_K) return mmq_launch<T_Q5_K>(gateup, tt, nw, items, a, st), true;
  return false;
}

}  // namespace zm
