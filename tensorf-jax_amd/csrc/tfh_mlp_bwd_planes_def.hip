// Launches of k_mlp_bwd_planes for the 24-channel, 6-frequency shape.
#include "tfh_mlp_bwd_planes.h"

namespace tfh {

int32_t launch_bwd_planes_def(bool bf, const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  if (bf)
    return a.ncam > 0 ? run_planes<BwdDef, 1, true, false, false>(w, a, st)
                      : run_planes<BwdDef, 1, false, false, true>(w, a, st);
  return a.ncam > 0 ? run_planes<BwdDef, 3, true, false, false>(w, a, st)
                    : run_planes<BwdDef, 3, false, false, false>(w, a, st);
}

}  // namespace tfh
