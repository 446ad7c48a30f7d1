// One translation unit per (dtype, GEMM kind, reduction tail): compiled with -DGMLP_DT=<0|1>
// -DGMLP_KIND=<0..6> -DGMLP_KT=<0|1> so the kernels build in parallel.  Each unit instantiates
// every tile class; GMLP_KT=1 are the kernels for reduction lengths that are not a multiple of 64
// (kinds with a reduction-contiguous operand, all but 4), which have no predicated class.
#include "gemm_pipelined.hpp"
#include "launch.hpp"

namespace gmlp {

#if GMLP_DT == 0
typedef f16 DT;
#else
typedef bf16 DT;
#endif

constexpr bool KT = GMLP_KT;

#define GMLP_LARGE(AKS, BKS, NB, EPI, BN_L) \
  launch_gemm_pipelined<DT, 256, BN_L, 16, 2, 2, AKS, BKS, NB, EPI<DT>, KT>
#define GMLP_MEDIUM(AKS, BKS, NB, EPI, BN_M) \
  launch_gemm_pipelined<DT, 128, BN_M, 16, 2, 2, AKS, BKS, NB, EPI<DT>, KT>
// (WN: wavefronts side by side, 2 or 4.  A tile's epilogue is a chain of loads, conversions and stores per
// wavefront: eight wavefronts halve it where it is long, at up to 43 % more LDS reads in the loop.  Plain stores and
// partial sums: no difference; dH: WIDE 1 % at most, no registers for it on TALL.  Gate/up: gate_up_eight_wavefronts.)
#define GMLP_TALL(AKS, BKS, NB, EPI, BN_T, WN) \
  launch_gemm_pipelined<DT, 192, BN_T, 16, 2, WN, AKS, BKS, NB, EPI<DT>, KT>
#define GMLP_WIDE(AKS, BKS, NB, EPI, BN_W, WN) \
  launch_gemm_pipelined<DT, 128, BN_W, 16, 2, WN, AKS, BKS, NB, EPI<DT>, KT>
#define GMLP_LARGE_GROUP \
  launch_gemm_group_pipelined<DT, 256, 256, 16, 2, 2, true, true, 1, EpiStore<DT>>
#define GMLP_MEDIUM_GROUP \
  launch_gemm_group_pipelined<DT, 128, 128, 16, 2, 2, true, true, 1, EpiStore<DT>>

#define GMLP_DISPATCH(AKS, BKS, NB, EPI, BN_L, BN_M, WN_W, WN_T)                                 \
  if (tile_class == TILE_LARGE) return GMLP_LARGE(AKS, BKS, NB, EPI, BN_L)(ga, ea, s);           \
  if constexpr (!(AKS)) {                                                                        \
    if (tile_class == TILE_WIDE) return GMLP_WIDE(AKS, BKS, NB, EPI, BN_L, WN_W)(ga, ea, s);     \
    if (tile_class == TILE_TALL) return GMLP_TALL(AKS, BKS, NB, EPI, BN_L, WN_T)(ga, ea, s);     \
  }                                                                                              \
  if (tile_class == TILE_MEDIUM_FULL) return GMLP_MEDIUM(AKS, BKS, NB, EPI, BN_M)(ga, ea, s);    \
  if constexpr (KT) return hipErrorInvalidValue; /* launch.hpp sends it to the other unit */       \
  else return launch_gemm<DT, 128, BN_M, 64, 2, 2, AKS, BKS, NB, true, EPI<DT>>(ga, ea, s);

#if GMLP_KIND == 0
// Gate/up on TALL tiles: the shorter epilogue of eight wavefronts against their slower loop, by the reduction's
// length.  Time with four over eight by the number of 64-wide reduction tiles, weights from memory / from cache (geometric
// means over 1396 launches of random shapes):
//                          8..11        12..15       16..19       20..23       28..31       32..35       48..55       96 on
//   SiLU (packed)      1.07 / 1.08  1.02 / 1.05  0.98 / 1.03  0.96 / 1.02  0.94 / 1.01  0.93 / 1.00  0.91 / 0.98  0.89 / 0.90
//   other activations  1.13 / 1.14  1.07 / 1.10  1.02 / 1.08  1.00 / 1.06  0.97 / 1.04  0.95 / 1.03  0.93 / 1.00  0.91 / 0.90
// The lines are about where what eight lose from memory (a model's layers come by in turn, and its weights with them) outweighs
// what they gain from cache (one layer called over and over).  us, eight -> four: M=3582, K=3200, N=11992 G and U kept 518 ->
// 482; M=1357, K=1160, N=3096 gelu stays on eight (37.3 with four, 34.3).  On WIDE tiles eight are never behind (1.03 at 20
// tiles, 1.00 from 96 on).
template <typename Epi>
static bool gate_up_eight_wavefronts(const GemmArgs& ga) {
  return ga.K <= 64 * (std::is_same<Epi, EpiGateUpPacked<DT>>::value ? 15 : 31);
}
template <>
hipError_t launch_gateup_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiGateUp<DT>::Args& ea,
                             hipStream_t s) {
  // the usual case (SiLU, no keep-mask output) has kernels of its own, see EpiGateUpPacked
  if (EpiGateUpPacked<DT>::packed_eligible(ea)) {
    if (tile_class == TILE_LARGE) return GMLP_LARGE(false, false, 2, EpiGateUpPacked, 128)(ga, ea, s);
    if (tile_class == TILE_WIDE) return GMLP_WIDE(false, false, 2, EpiGateUpPacked, 128, 4)(ga, ea, s);
    if (tile_class == TILE_TALL)
      return gate_up_eight_wavefronts<EpiGateUpPacked<DT>>(ga) ? GMLP_TALL(false, false, 2, EpiGateUpPacked, 128, 4)(ga, ea, s)
                                                               : GMLP_TALL(false, false, 2, EpiGateUpPacked, 128, 2)(ga, ea, s);
    if (tile_class == TILE_MEDIUM_FULL) return GMLP_MEDIUM(false, false, 2, EpiGateUpPacked, 64)(ga, ea, s);
  }
  if (tile_class == TILE_TALL && gate_up_eight_wavefronts<EpiGateUp<DT>>(ga))
    return GMLP_TALL(false, false, 2, EpiGateUp, 128, 4)(ga, ea, s);
  GMLP_DISPATCH(false, false, 2, EpiGateUp, 128, 64, 4, 2)
}
template <>
hipError_t launch_gateup_split_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiPartial<DT>::Args& ea, hipStream_t s) {
  if (tile_class == TILE_WIDE) return GMLP_WIDE(false, false, 2, EpiPartial, 128, 2)(ga, ea, s);
  return launch_gemm_pipelined<DT, 128, 64, 16, 2, 2, false, false, 2, EpiPartial<DT>, KT>(ga, ea, s);
}
#elif GMLP_KIND == 1
template <>
hipError_t launch_linear_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiStore<DT>::Args& ea,
                             hipStream_t s) {
  GMLP_DISPATCH(false, false, 1, EpiStore, 256, 128, 2, 2)
}
template <>
hipError_t launch_linear_split_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiPartial<DT>::Args& ea, hipStream_t s) {
  if (tile_class == TILE_WIDE) return GMLP_WIDE(false, false, 1, EpiPartial, 256, 2)(ga, ea, s);
  return launch_gemm_pipelined<DT, 128, 128, 16, 2, 2, false, false, 1, EpiPartial<DT>, KT>(ga, ea, s);
}
#elif GMLP_KIND == 2
template <>
hipError_t launch_dh_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiDh<DT>::Args& ea,
                         hipStream_t s) {
  GMLP_DISPATCH(false, true, 1, EpiDh, 256, 128, 4, 2)
}
#elif GMLP_KIND == 3
template <>
hipError_t launch_dx_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiStore<DT>::Args& ea,
                         hipStream_t s) {
  GMLP_DISPATCH(false, true, 1, EpiStore, 256, 128, 2, 2)
}
template <>
hipError_t launch_dx_split_kt<DT, KT>(int tile_class, const GemmArgs& ga, const EpiPartial<DT>::Args& ea, hipStream_t s) {
  if (tile_class == TILE_WIDE) return GMLP_WIDE(false, true, 1, EpiPartial, 256, 2)(ga, ea, s);
  return launch_gemm_pipelined<DT, 128, 128, 16, 2, 2, false, true, 1, EpiPartial<DT>, KT>(ga, ea, s);
}
#elif GMLP_KIND == 4
template <>
hipError_t launch_dw<DT>(int tile_class, const GemmArgs& ga, const EpiStore<DT>::Args& ea,
                         hipStream_t s) {
  GMLP_DISPATCH(true, true, 1, EpiStore, 256, 128, 2, 2)
}
template <>
hipError_t launch_dw_group<DT>(int tile_class, GemmGroup<EpiStore<DT>::Args>& grp, hipStream_t s) {
  return tile_class == TILE_LARGE ? GMLP_LARGE_GROUP(grp, s) : GMLP_MEDIUM_GROUP(grp, s);
}
template <>
hipError_t launch_dw_group_split<DT>(int, GemmGroup<EpiPartial<DT>::Args>& grp, hipStream_t s) {
  return launch_gemm_group_pipelined<DT, 128, 128, 16, 2, 2, true, true, 1, EpiPartial<DT>>(grp, s);
}
#elif GMLP_KIND == 5
template <>
hipError_t launch_dx_dw_kt<DT, KT>(int x_class, DxDwGroup<DT, EpiStore<DT>>& grp, bool dx_first, hipStream_t s) {
  if (x_class == TILE_LARGE) return launch_dx_dw_pipelined<DT, 256, 256, 256, KT>(grp, dx_first, s);
  if (x_class == TILE_TALL) return launch_dx_dw_pipelined<DT, 192, 256, 256, KT>(grp, dx_first, s);
  if (x_class == TILE_WIDE) return launch_dx_dw_pipelined<DT, 128, 256, 256, KT>(grp, dx_first, s);
  return launch_dx_dw_pipelined<DT, 128, 128, 128, KT>(grp, dx_first, s);
}
template <>
hipError_t launch_dx_dw_kt<DT, KT>(int, DxDwGroup<DT, EpiStore<DT>, EpiPartial<DT>>& grp, bool dx_first, hipStream_t s) {
  return launch_dx_dw_pipelined<DT, 128, 128, 128, KT>(grp, dx_first, s);
}
#elif GMLP_KIND == 6
template <>
hipError_t launch_dx_dw_kt<DT, KT>(int x_class, DxDwGroup<DT, EpiPartial<DT>>& grp, bool dx_first, hipStream_t s) {
  if (x_class == TILE_LARGE) return launch_dx_dw_pipelined<DT, 256, 256, 256, KT>(grp, dx_first, s);
  if (x_class == TILE_WIDE) return launch_dx_dw_pipelined<DT, 128, 256, 256, KT>(grp, dx_first, s);
  return launch_dx_dw_pipelined<DT, 128, 128, 128, KT>(grp, dx_first, s);
}
template <>
hipError_t launch_dx_dw_kt<DT, KT>(int, DxDwGroup<DT, EpiPartial<DT>, EpiPartial<DT>>& grp, bool dx_first, hipStream_t s) {
  return launch_dx_dw_pipelined<DT, 128, 128, 128, KT>(grp, dx_first, s);
}
#endif

}  // namespace gmlp
