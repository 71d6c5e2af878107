// The forces pass of kernels_forces.hpp with Akinci tension.
#include "kernels_forces.hpp"

namespace cryo {

void launch_forces_akinci(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                   bool continuity, bool thermal, int lanes, hipStream_t s) {
  launch_forces_model<2>(pv, g, P, L, st, n, continuity, thermal, lanes, s);
}

}  // namespace cryo
