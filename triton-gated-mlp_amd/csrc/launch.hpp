// Host-side launch interface between the C ABI (api.hip) and the kernel translation units.
#pragma once
#include "colsum.hpp"
#include "gemm.hpp"
#include "gemm_tiles.hpp"

namespace gmlp {

// Tile classes (four wavefronts per workgroup, eight of half the width where said; 64-wide reduction tiles).
//   LARGE        256x256 output tiles, wavefronts of 128x128, pipelined kernel
//   WIDE         128x256 output tiles, wavefronts of 64x128 (gate/up without a split, dH: eight of 64x64), pipelined kernel
//                (not the weight gradients):
//                one workgroup per CU, three ring entries of both operands.  Half of LARGE's work per
//                workgroup at 5/6 of its throughput: for grids that LARGE fills badly and for short
//                batches, where it reads the weights once per 128 token rows from L2 and needs fewer
//                splits than MEDIUM_FULL
//   TALL         192x256 output tiles, wavefronts of 96x128 (gate/up with a short reduction: eight of 96x64), pipelined
//                kernel (not the weight gradients, no split reductions): three quarters of LARGE's work, for grids that
//                LARGE fills badly
//   MEDIUM_FULL  128x128 output tiles, wavefronts of 64x64, pipelined kernel; two workgroups per CU,
//                for problems with too few 256x256 tiles to fill the chip
//   MEDIUM       128x128, predicated register-staged kernel, 64-bit addresses: operands too large for
//                the pipelined kernels' 32-bit byte offsets
//   F32_*        the float32 kernel's tiles (gemm_f32.hip): 128 x 128 or 64 x 64; with two accumulator
//                sets 128 x 64 or 64 x 64; HALVES: 64 x 64, one workgroup for both halves of a down projection's reduction
enum TileClass { TILE_LARGE = 0, TILE_MEDIUM = 1, TILE_MEDIUM_FULL = 2, TILE_F32_128 = 3, TILE_F32_64 = 4, TILE_WIDE = 5,
                 TILE_TALL = 6, TILE_F32_HALVES = 7 };

// kinds of GEMM the gated MLP needs; each is instantiated per dtype and tile class, and for reduction
// lengths that are (KT = false) or are not a multiple of 64, the width of a reduction tile.
template <typename T, bool KT>
hipError_t launch_gateup_kt(int tile_class, const GemmArgs& ga, const typename EpiGateUp<T>::Args& ea,
                            hipStream_t s);  // A KC, B KC, two accumulator sets
template <typename T, bool KT>
hipError_t launch_linear_kt(int tile_class, const GemmArgs& ga, const typename EpiStore<T>::Args& ea,
                            hipStream_t s);  // A KC, B KC
template <typename T, bool KT>
hipError_t launch_dh_kt(int tile_class, const GemmArgs& ga, const typename EpiDh<T>::Args& ea,
                        hipStream_t s);  // A KC, B KS
template <typename T, bool KT>
hipError_t launch_dx_kt(int tile_class, const GemmArgs& ga, const typename EpiStore<T>::Args& ea,
                        hipStream_t s);  // A KC, B KS, two reduction segments
// Split-reduction variants (128x128 tiles): partial sums to a fp32 workspace, see splitk_reduce.
template <typename T, bool KT>
hipError_t launch_linear_split_kt(int tile_class, const GemmArgs& ga, const typename EpiPartial<T>::Args& ea, hipStream_t s);
template <typename T, bool KT>
hipError_t launch_dx_split_kt(int tile_class, const GemmArgs& ga, const typename EpiPartial<T>::Args& ea, hipStream_t s);
template <typename T, bool KT>
hipError_t launch_gateup_split_kt(int tile_class, const GemmArgs& ga, const typename EpiPartial<T>::Args& ea, hipStream_t s);

// The predicated class (and float32) has one kernel for every reduction length.
template <typename T>
bool reduction_tail(int tile_class, const GemmArgs& ga) {
  return !std::is_same<T, float>::value && tile_class != TILE_MEDIUM && ga.K % 64 != 0;
}
#define GMLP_BY_TAIL(KIND, EPI)                                                                              \
  template <typename T>                                                                                      \
  hipError_t launch_##KIND(int tile_class, const GemmArgs& ga, const typename EPI<T>::Args& ea, hipStream_t s) { \
    if constexpr (!std::is_same<T, float>::value)                                                            \
      if (reduction_tail<T>(tile_class, ga)) return launch_##KIND##_kt<T, true>(tile_class, ga, ea, s);        \
    return launch_##KIND##_kt<T, false>(tile_class, ga, ea, s);                                              \
  }
#define GMLP_SPLIT_BY_TAIL(KIND)                                                                             \
  template <typename T>                                                                                      \
  hipError_t launch_##KIND##_split(int tile_class, const GemmArgs& ga, const typename EpiPartial<T>::Args& ea,  \
                                   hipStream_t s) {                                                          \
    if constexpr (!std::is_same<T, float>::value)                                                            \
      if (reduction_tail<T>(tile_class, ga)) return launch_##KIND##_split_kt<T, true>(tile_class, ga, ea, s);  \
    return launch_##KIND##_split_kt<T, false>(tile_class, ga, ea, s);                                        \
  }
GMLP_BY_TAIL(gateup, EpiGateUp)
GMLP_BY_TAIL(linear, EpiStore)
GMLP_BY_TAIL(dh, EpiDh)
GMLP_BY_TAIL(dx, EpiStore)
GMLP_SPLIT_BY_TAIL(gateup)
GMLP_SPLIT_BY_TAIL(linear)
GMLP_SPLIT_BY_TAIL(dx)
#undef GMLP_BY_TAIL
#undef GMLP_SPLIT_BY_TAIL

template <typename T>
hipError_t launch_dw(int tile_class, const GemmArgs& ga, const typename EpiStore<T>::Args& ea,
                     hipStream_t s);  // A KS, B KS

// Several weight-gradient GEMMs of one tile class (LARGE, MEDIUM_FULL or F32_*) as one grid.
template <typename T>
hipError_t launch_dw_group(int tile_class, GemmGroup<typename EpiStore<T>::Args>& grp, hipStream_t s);

// The same with a split reduction (on MEDIUM_FULL, F32_128 or F32_64): every problem's ga.splits partial sums,
// then their totals.
template <typename T>
hipError_t launch_dw_group_split(int tile_class, GemmGroup<typename EpiPartial<T>::Args>& grp, hipStream_t s);
template <typename T>
struct ReduceGroup {
  const float* ws[GEMM_GROUP_MAX + 1];
  T* out[GEMM_GROUP_MAX + 1];
  size_t n[GEMM_GROUP_MAX + 1];  // elements of an output, and between consecutive splits
  int splits[GEMM_GROUP_MAX + 1];
  int count;
};
template <typename T>
hipError_t launch_splitk_reduce_group(const ReduceGroup<T>& g, hipStream_t s);

// dX and up to three weight gradients as one grid: dX on `x_class` (LARGE, TALL, WIDE beside large tiles of
// the weight gradients, MEDIUM_FULL beside MEDIUM_FULL ones; a split dX, EpiPartial, not TALL; split weight
// gradients MEDIUM_FULL beside MEDIUM_FULL).
// The workgroups of the problem that takes longer per tile should come first.
template <typename T, bool KT>
hipError_t launch_dx_dw_kt(int x_class, DxDwGroup<T, EpiStore<T>>& grp, bool dx_first, hipStream_t s);
template <typename T, bool KT>
hipError_t launch_dx_dw_kt(int x_class, DxDwGroup<T, EpiPartial<T>>& grp, bool dx_first, hipStream_t s);
template <typename T, bool KT>
hipError_t launch_dx_dw_kt(int x_class, DxDwGroup<T, EpiStore<T>, EpiPartial<T>>& grp, bool dx_first, hipStream_t s);
template <typename T, bool KT>
hipError_t launch_dx_dw_kt(int x_class, DxDwGroup<T, EpiPartial<T>, EpiPartial<T>>& grp, bool dx_first, hipStream_t s);

// Generic launcher used by the instantiation units.
template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool A_KS, bool B_KS, int NB,
          bool EDGE, typename Epi>
hipError_t launch_gemm(const GemmArgs& ga, const typename Epi::Args& ea, hipStream_t s) {
  typedef GemmConfig<T, BM, BN, BK, WGM, WGN, A_KS, B_KS, NB, EDGE> Cfg;
  constexpr auto kern = gemm_kernel<T, BM, BN, BK, WGM, WGN, A_KS, B_KS, NB, EDGE, Epi>;
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, Cfg::LDS_BYTES>, s)) return e;
  int tiles_m = (ga.M + BM - 1) / BM, tiles_n = (ga.N + BN - 1) / BN;
  dim3 grid(tiles_m * tiles_n), block(Cfg::NT);
  hipLaunchKernelGGL(kern, grid, block, Cfg::LDS_BYTES, s, ga, ea);
  return hipGetLastError();
}

// decode.hip
template <typename T>
hipError_t launch_decode(const T* x, const T* wg, const T* wu, const T* wd, const T* bg,
                         const T* bu, const T* bd, T* h, T* y, int M, int K, int N, int act,
                         hipStream_t s);

// decode_stream.hip: LDS-ring streaming variant for K and N from 768 up, any multiples of 8
bool decode_stream_supported(int M, int K, int N);
template <typename T>
hipError_t launch_decode_stream(const T* x, const T* wg, const T* wu, const T* wd, const T* bg,
                                const T* bu, const T* bd, T* h, T* y, int M, int K, int N,
                                int act, hipStream_t s);

// aux.hip
template <typename T>
hipError_t launch_gating_bwd(const T* dh, const T* g, const T* u, T* dg, T* du, int64_t M, int64_t N,
                             int act, const DropoutParams& d, hipStream_t s);
// Second stage of a split reduction: Epi (EpiStore or EpiGateUp) applied to
// sum_s ws[s*split_stride (+ acc_stride) + m*N + n].
template <typename T, typename Epi>
hipError_t launch_splitk_reduce(const float* ws, int splits, size_t split_stride, size_t acc_stride,
                                const typename Epi::Args& ea, int64_t M, int64_t N, hipStream_t s);
template <typename T>
hipError_t launch_colsum_group(const ColsumGroup<T>& g, int count, int64_t M, hipStream_t s);
size_t colsum_workspace_bytes(int64_t M, int64_t C);
// Column sums of one array with the first stage's partial sums in a static device array of the
// library (no workspace argument, no allocation); C <= COLSUM_STATIC_MAX_C.
constexpr int64_t COLSUM_STATIC_MAX_C = 32768;
// Address of that array on the current device; the first call on a device looks the symbol up
// and refuses to while `s` is capturing.
hipError_t colsum_static_scratch(float** out, hipStream_t s);
template <typename T>
hipError_t launch_colsum_static(const T* a, T* out, int64_t M, int64_t C, hipStream_t s);
hipError_t launch_dropout_mask(uint8_t* mask, int64_t M, int64_t N, const DropoutParams& d,
                               hipStream_t s);

}  // namespace gmlp
