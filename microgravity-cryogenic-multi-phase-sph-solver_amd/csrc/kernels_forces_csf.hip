// The forces pass of kernels_forces.hpp with CSF tension with vapour present.
#include "kernels_forces.hpp"

namespace cryo {

void launch_forces_csf(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                   bool continuity, bool thermal, int lanes, hipStream_t s) {
  launch_forces_model<1>(pv, g, P, L, st, n, continuity, thermal, lanes, s);
}

}  // namespace cryo
