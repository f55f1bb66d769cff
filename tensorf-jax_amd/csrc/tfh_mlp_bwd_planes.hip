// Launches of k_mlp_bwd_planes for the fused training steps of the 48-channel,
// 2-frequency shape, and the operand tables.
#include "tfh_mlp_bwd_planes.h"

namespace tfh {

size_t bwd_planes_table_bytes(BwdKind kind, bool bf) {
  const int total = kind == BwdKind::kStd ? BwdTables<BwdStd>::total : BwdTables<BwdDef>::total;
  return align_up((size_t)total * 2 * (bf ? 1 : 3), 256);
}

int bwd_planes_pack_flags(BwdKind kind) {
  return (kind == BwdKind::kStd ? BwdTables<BwdStd>::total : BwdTables<BwdDef>::total) /
         kPackThreads;
}

int32_t pack_bwd_planes(BwdKind kind, bool bf, const MlpW& w, void* tables, int32_t* flags,
                        hipStream_t st) {
  return kind == BwdKind::kStd ? pack_planes<BwdStd>(bf, w, tables, flags, st)
                               : pack_planes<BwdDef>(bf, w, tables, flags, st);
}

int32_t launch_bwd_planes_train(bool bf, const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  if (bf)
    return a.ncam > 0 ? run_planes<BwdStd, 1, true, true, true>(w, a, st)
                      : run_planes<BwdStd, 1, false, true, true>(w, a, st);
  return a.ncam > 0 ? run_planes<BwdStd, 3, true, true, false>(w, a, st)
                    : run_planes<BwdStd, 3, false, true, false>(w, a, st);
}

}  // namespace tfh
