// The forces pass of kernels_forces.hpp with no tension model.
#include "kernels_forces.hpp"

namespace cryo {

void launch_forces_none(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                   bool continuity, bool thermal, int lanes, hipStream_t s) {
  launch_forces_model<0>(pv, g, P, L, st, n, continuity, thermal, lanes, s);
}

}  // namespace cryo
