// Launches of k_mlp_bwd_planes, in a translation unit of its own (register
// allocation, see tfh_mlp_kernels.h).
#include "tfh_mlp_bwd_planes.h"

namespace tfh {

template <class SH, int NP, bool FILM, bool SPLIT0>
static int32_t run_planes(const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  using L = BwdLds<SH, NP>;
  static_assert(L::bytes <= 160 * 1024, "the tile fits the LDS of a CU");
  __bf16* tables = static_cast<__bf16*>(a.tables);
  hipLaunchKernelGGL((k_pack_bwd<SH, NP>), dim3((BwdTables<SH>::total + 255) / 256), dim3(256), 0,
                     st, w, tables);
  TFH_TRY(check_launch("mlp bwd: operand tables"));
  auto kernel = k_mlp_bwd_planes<SH, NP, FILM, SPLIT0>;
  allow_lds(kernel, L::bytes);
  hipLaunchKernelGGL(kernel, dim3(a.nblk), dim3(512), L::bytes, st, w, tables, a.feats, a.dirs,
                     a.grgb, a.M, a.rpr, a.gfeat, a.partials, a.gp, a.act, a.rgb, a.cams,
                     a.gembed, a.ncam);
  return check_launch("mlp bwd");
}

size_t bwd_planes_table_bytes(bool bf) {
  return align_up((size_t)BwdTables<BwdStd>::total * 2 * (bf ? 1 : 3), 256);
}

int bwd_planes_tile_rows(bool bf) { return bf ? BwdLds<BwdStd, 1>::TM : BwdLds<BwdStd, 3>::TM; }

int32_t launch_bwd_planes(bool bf, const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  if (bf)
    return a.ncam > 0 ? run_planes<BwdStd, 1, true, true>(w, a, st)
                      : run_planes<BwdStd, 1, false, true>(w, a, st);
  return a.ncam > 0 ? run_planes<BwdStd, 3, true, true>(w, a, st)
                    : run_planes<BwdStd, 3, false, true>(w, a, st);
}

}  // namespace tfh
