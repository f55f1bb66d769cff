// Launches of k_mlp_bwd_planes for the 48-channel, 2-frequency shape where the
// backward keeps the activations itself (callers other than the fused steps).
#include "tfh_mlp_bwd_planes.h"

namespace tfh {

int32_t launch_bwd_planes_std(bool bf, const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  if (bf)
    return a.ncam > 0 ? run_planes<BwdStd, 1, true, false, false>(w, a, st)
                      : run_planes<BwdStd, 1, false, false, true>(w, a, st);
  return a.ncam > 0 ? run_planes<BwdStd, 3, true, false, false>(w, a, st)
                    : run_planes<BwdStd, 3, false, false, false>(w, a, st);
}

}  // namespace tfh
