// float32 path: the same six GEMMs and fused epilogues on v_mfma_f32_32x32x2_f32, for callers that
// keep the module in float32 (as the reference's own tests do).
//
// Bound: the matrix cores (157 TFLOP/s; one 32x32x2 MFMA takes 64 clocks, so operand traffic is an
// eighth of what the 16-bit kernels move per clock and plain staging keeps up).  What decides is how
// evenly the output tiles spread over the compute units: a CU runs several workgroups of 4
// wavefronts (2 x 2) at once, and the launch takes as long as the CU with the most tiles.  Hence
// three tile shapes and a split reduction, chosen by estimated time (plan_f32 in api.hip), and the
// weight gradients of a pass in one grid.
//
// A reduction tile is BK = 32 elements (16 for the 128-row tiles).  It moves global memory -> LDS
// without passing through registers (global_load_lds: the next tiles' loads stay in flight while the
// MFMAs of the current one run) into a ring of NS stages, one barrier per reduction tile.  Depth is
// what counts: operands that L2 does not hold take longer to arrive than a tile takes to compute.
// A lane's LDS position is fixed by the transfer (wave base + 16 bytes x lane), so the layouts below
// are made by choosing WHICH 16-byte chunk a lane fetches.
//   KC tiles ([row][k]): chunk c of row r at position c ^ swz(r): 16 consecutive rows x one chunk
//     cover all 64 banks, so fragments are read with ds_read_b128, 4 reduction elements at a time.
//     Which two k an MFMA multiplies is free as long as both operands agree: in step s it takes
//     k = 8 s + 4 (lane / 32) + j, j = 0..3.
//   KS tiles ([k][row]): row index XORed with 32 for every other group of 4 k, so that the two
//     halves of a wavefront, 4 k apart, read different banks.
#include "launch.hpp"
#include "lds_dma.hpp"

namespace gmlp {

// What the chunks beyond the end of a reduction are fetched from.
static __device__ __align__(16) float f32_zeros[4];

__device__ __forceinline__ void global16_to_lds(const float* p, uint32_t lds_wave_base) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds_wave_base), "v"(p)
      : "memory");
}

template <int ROWS, int BK, bool KS>
struct F32Tile {
  static constexpr int BYTES = ROWS * BK * 4;
  static constexpr int LOADS = BYTES / 1024 / 4;  // per wavefront and tile
  static_assert(BK == 16 || BK == 32, "reduction tiles of 16 or 32");
  static_assert(LOADS >= 1, "every wavefront loads");

  const float* ptr[LOADS];  // this lane's 16-byte chunks of the tile the pointers stand at

  static __device__ __forceinline__ int swz(int r) { return BK == 32 ? (r >> 1) & 7 : (r >> 2) & 3; }
  // Row (first of 4 for KS) and reduction index, within the tile, of the chunk that load i fetches.
  static __device__ __forceinline__ void chunk_of(int i, int wave, int lane, int& r, int& k) {
    const int q = (wave * LOADS + i) * 64 + lane;  // 16-byte position in the tile
    if (KS) {
      k = q / (ROWS / 4);
      r = ((q % (ROWS / 4)) * 4) ^ (((k >> 2) & 1) << 5);
    } else {
      r = q / (BK / 4);
      k = ((q % (BK / 4)) ^ swz(r)) * 4;
    }
  }
  // Rows (columns of a KS tile) beyond the matrix read the last valid ones: they only feed output
  // elements that are not stored.
  __device__ __forceinline__ void start(const float* __restrict__ p, int ld, int r0, int k0, int rtot, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int r, k;
      chunk_of(i, wave, lane, r, k);
      r = min(r0 + r, KS ? rtot - 4 : rtot - 1);
      ptr[i] = KS ? p + (size_t)(k0 + k) * ld + r : p + (size_t)r * ld + (k0 + k);
    }
  }
  // Issues the tile's loads into the stage at LDS address `lds` and moves on to the next tile.
  // kleft: reduction elements left from the tile's start; chunks beyond them read zeros.
  __device__ __forceinline__ void fetch(uint32_t lds, int ld, int kleft, int wave, int lane) {
    const size_t step = KS ? (size_t)BK * ld : (size_t)BK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int r, k;
      chunk_of(i, wave, lane, r, k);
      global16_to_lds(k < kleft ? ptr[i] : f32_zeros, lds + (wave * LOADS + i) * 1024);
      ptr[i] += step;
    }
  }
  // The four reduction elements step s gives this lane, of the 32 rows starting at `row0`.
  static __device__ __forceinline__ f32x4 frag(const float* lds, int row0, int s, int lane) {
    const int r = row0 + (lane & 31), h = lane >> 5;
    if (KS) {
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = lds[(8 * s + 4 * h + j) * ROWS + (r ^ (h << 5))];
      return v;
    }
    return *(const f32x4*)(lds + r * BK + (((2 * s + h) ^ swz(r)) << 2));
  }
};

template <int BM, int BN, bool A_KS, bool B_KS, int NB>
struct F32Config {
  static constexpr int BK = BM == 128 ? 16 : 32;
  static constexpr int NS = BM == 128 ? 4 : 3;
  typedef F32Tile<BM, BK, A_KS> AT;
  typedef F32Tile<BN, BK, B_KS> BT;
  static constexpr int STAGE = AT::BYTES + NB * BT::BYTES;
  static constexpr int LOADS = AT::LOADS + NB * BT::LOADS;
  static constexpr int LDS_BYTES = NS * STAGE;
};

template <int BM, int BN, bool A_KS, bool B_KS, int NB, typename Epi>
__device__ __forceinline__ void gemm_f32_body(const GemmArgs& ga, typename Epi::Args ea, int pid, int nwg) {
  typedef F32Config<BM, BN, A_KS, B_KS, NB> Cfg;
  typedef typename Cfg::AT AT;
  typedef typename Cfg::BT BT;
  constexpr int BK = Cfg::BK, NS = Cfg::NS, STAGE = Cfg::STAGE;
  constexpr int TM = BM / 64, TN = BN / 64;  // 32x32 MFMA tiles per wavefront
  static_assert(TM >= 1 && TN >= 1, "wavefronts own at least one MFMA tile");
  extern __shared__ __align__(1024) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void*)smem;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_m = (ga.M + BM - 1) / BM, tiles_n = (ga.N + BN - 1) / BN, ntiles = tiles_m * tiles_n;
  const int u = xcd_contiguous(pid, nwg, ga.nxcd);
  const int split = Epi::SPLIT ? u / ntiles : 0;
  int tm_i, tn_i;
  tile_of_grouped(u - split * ntiles, tiles_m, tiles_n, ga.group_m, tm_i, tn_i);
  const int m0 = tm_i * BM, n0 = tn_i * BN;
  if constexpr (Epi::SPLIT) ea.ws += (size_t)split * ea.split_stride;

  const int kt_seg = (ga.K + BK - 1) / BK, kt_all = kt_seg * ga.nseg;
  int kt_first = 0, kt_end = kt_all;
  if constexpr (Epi::SPLIT) {
    const int per = (kt_all + ga.splits - 1) / ga.splits;
    kt_first = min(split * per, kt_all);
    kt_end = min(kt_first + per, kt_all);
  }

  f32x16 acc[NB][TM][TN];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][i][j][r] = 0.f;

  AT at;
  BT bt[NB];
  int seg = kt_first >= kt_seg ? 1 : 0, kleft = 0;
  auto start = [&](int kk) __attribute__((always_inline)) {
    at.start((const float*)ga.A[seg], ga.lda, m0, kk * BK, ga.M, wave, lane);
#pragma unroll
    for (int b = 0; b < NB; ++b)
      bt[b].start((const float*)ga.B[NB == 2 ? b : seg], ga.ldb, n0, kk * BK, ga.N, wave, lane);
    kleft = ga.K - kk * BK;
  };
  // The next tile in reduction order into ring stage `st` (beyond the last one: zeros).
  auto fetch = [&](int st) __attribute__((always_inline)) {
    if (NB == 1 && kleft <= 0 && seg + 1 < ga.nseg) {  // on into the second reduction segment
      seg = 1;
      start(0);
    }
    const uint32_t lds = lds_base + st * STAGE;
    at.fetch(lds, ga.lda, kleft, wave, lane);
#pragma unroll
    for (int b = 0; b < NB; ++b) bt[b].fetch(lds + AT::BYTES + b * BT::BYTES, ga.ldb, kleft, wave, lane);
    kleft -= BK;
  };

  // Fragments are read one step ahead of their MFMAs, across tiles too: before a tile's last step the
  // wavefronts meet at the tile's only barrier, after which the next tile may be read and the stage of
  // the current one (every fragment of it has been read) takes the tile NS further on.
  constexpr int STEPS = BK / 8;
  static_assert(STEPS % 2 == 0, "fragment registers alternate by step and every tile starts on the first");
  f32x4 av[2][TM], bv[2][NB][TN];
  auto read = [&](int st, int ks) __attribute__((always_inline)) {
    const float* s = (const float*)(smem + st * STAGE);
#pragma unroll
    for (int i = 0; i < TM; ++i) av[ks & 1][i] = AT::frag(s, wm * (BM / 2) + i * 32, ks, lane);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bv[ks & 1][b][j] = BT::frag(s + (AT::BYTES + b * BT::BYTES) / 4, wn * (BN / 2) + j * 32, ks, lane);
  };

  start(kt_first - seg * kt_seg);
#pragma unroll
  for (int p = 0; p < NS; ++p) fetch(p);
  wait_vmem<(NS - 1) * Cfg::LOADS>();
  __syncthreads();
  read(0, 0);
  int st = 0;  // ring stage of tile kt
  for (int kt = kt_first; kt < kt_end; ++kt) {
    const int st_next = st + 1 == NS ? 0 : st + 1;
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks) {
      if (ks + 1 < STEPS) {
        read(st, ks + 1);
      } else {
        wait_vmem<(NS - 2) * Cfg::LOADS>();  // all but the youngest NS - 2 tiles: tile kt + 1 has landed
        __syncthreads();
        read(st_next, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              // operands swapped: a lane ends up with 4 consecutive output columns of one row
              acc[b][i][j] =
                  __builtin_amdgcn_mfma_f32_32x32x2f32(bv[ks & 1][b][j][e], av[ks & 1][i][e], acc[b][i][j], 0, 0, 0);
        if (e == 0 && ks + 1 == STEPS) {  // behind MFMAs that cover the address arithmetic
          __builtin_amdgcn_sched_barrier(0);
          fetch(st);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    st = st_next;
  }
  wait_vmem<0>();  // nothing may land in LDS after the workgroup has given it back

  // Epilogue, one 32x32 block at a time: an MFMA leaves a lane 4 consecutive columns of one row in 4
  // places, so stores straight from the accumulators would touch 32 bytes in each of 32 rows.  The
  // block goes through a wavefront-private LDS slab instead (rows of 36 floats: conflict-free), after
  // which 8 lanes share the 128 bytes of a row.  What the epilogue reads (G and U of dH) is in flight
  // meanwhile.
  __syncthreads();  // the slabs overwrite the ring
  constexpr int SLAB = 32 * 36;
  static_assert(4 * NB * SLAB * 4 <= Cfg::LDS_BYTES, "slabs fit the ring");
  float* slab = (float*)smem + wave * NB * SLAB;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row0 = m0 + wm * (BM / 2) + i * 32 + lane / 8;
      const int n = n0 + wn * (BN / 2) + j * 32 + (lane % 8) * 4;
      typename Epi::template Prefetch<4> pf[4];
      if (Epi::PREFETCH_DEPTH > 0) {
#pragma unroll
        for (int it = 0; it < 4; ++it)  // beyond the edge: the last valid elements, dropped below
          Epi::template prefetch<4>(ea, min(row0 + 8 * it, ga.M - 1), min(n, ga.N - 4), pf[it]);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *(f32x4*)(slab + b * SLAB + (lane & 31) * 36 + 8 * g + 4 * (lane >> 5)) =
              f32x4{acc[b][i][j][4 * g], acc[b][i][j][4 * g + 1], acc[b][i][j][4 * g + 2], acc[b][i][j][4 * g + 3]};
      // (same-wavefront LDS writes and reads are ordered)
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int m = row0 + 8 * it;
        const float* p = slab + (lane / 8 + 8 * it) * 36 + (lane % 8) * 4;
        alignas(16) float v0[4], v1[4];
        *(f32x4*)v0 = *(const f32x4*)p;
        *(f32x4*)v1 = *(const f32x4*)(p + (NB - 1) * SLAB);
        if (m < ga.M && n < ga.N) Epi::template apply<4, ACT_RUNTIME>(ea, m, n, v0, v1, pf[it]);
      }
    }
  }
}

template <int BM, int BN, bool A_KS, bool B_KS, int NB, typename Epi>
__global__ void __launch_bounds__(256) gemm_f32_kernel(GemmArgs ga, typename Epi::Args ea) {
  gemm_f32_body<BM, BN, A_KS, B_KS, NB, Epi>(ga, ea, blockIdx.x, gridDim.x);
}

template <int BM, int BN, typename Epi>
__global__ void __launch_bounds__(256) gemm_f32_group_kernel(GemmGroup<typename Epi::Args> grp) {
  int g = 0;
#pragma unroll
  for (int i = 1; i < GEMM_GROUP_MAX; ++i)
    if (i < grp.count && (int)blockIdx.x >= grp.first[i]) g = i;
  gemm_f32_body<BM, BN, true, true, 1, Epi>(grp.ga[g], grp.ea[g], (int)blockIdx.x - grp.first[g],
                                           grp.first[g + 1] - grp.first[g]);
}

template <int BM, int BN, bool A_KS, bool B_KS, int NB, typename Epi>
static hipError_t launch_f32_tile(const GemmArgs& ga, const typename Epi::Args& ea, hipStream_t s) {
  constexpr auto kern = gemm_f32_kernel<BM, BN, A_KS, B_KS, NB, Epi>;
  constexpr int LDS = F32Config<BM, BN, A_KS, B_KS, NB>::LDS_BYTES;
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, LDS>, s)) return e;
  const int tiles = ((ga.M + BM - 1) / BM) * ((ga.N + BN - 1) / BN);
  hipLaunchKernelGGL(kern, dim3(tiles * (Epi::SPLIT ? ga.splits : 1)), dim3(256), LDS, s, ga, ea);
  return hipGetLastError();
}
// One accumulator set: 128x128, 64x128 or 64x64 tiles; two: 128x64 or 64x64 (x 2).
template <bool A_KS, bool B_KS, int NB, typename Epi>
static hipError_t launch_f32(int tile_class, const GemmArgs& ga, const typename Epi::Args& ea, hipStream_t s) {
  if (tile_class == TILE_F32_128) return launch_f32_tile<128, 128 / NB, A_KS, B_KS, NB, Epi>(ga, ea, s);
  if constexpr (NB == 1)
    if (tile_class == TILE_F32_64X128) return launch_f32_tile<64, 128, A_KS, B_KS, NB, Epi>(ga, ea, s);
  return launch_f32_tile<64, 64, A_KS, B_KS, NB, Epi>(ga, ea, s);
}

template <>
hipError_t launch_gateup_kt<float, false>(int tc, const GemmArgs& ga, const EpiGateUp<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, false, 2, EpiGateUp<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_linear_kt<float, false>(int tc, const GemmArgs& ga, const EpiStore<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, false, 1, EpiStore<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_dh_kt<float, false>(int tc, const GemmArgs& ga, const EpiDh<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, true, 1, EpiDh<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_dx_kt<float, false>(int tc, const GemmArgs& ga, const EpiStore<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, true, 1, EpiStore<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_dw<float>(int, const GemmArgs&, const EpiStore<float>::Args&, hipStream_t) {
  return hipErrorInvalidValue;  // float32 weight gradients go through launch_dw_group
}
// Split reductions run on the smallest tile only (a grid of larger ones would be split further).
template <>
hipError_t launch_gateup_split_kt<float, false>(int, const GemmArgs& ga, const EpiPartial<float>::Args& ea, hipStream_t s) {
  return launch_f32_tile<64, 64, false, false, 2, EpiPartial<float>>(ga, ea, s);
}
template <>
hipError_t launch_linear_split_kt<float, false>(int, const GemmArgs&, const EpiPartial<float>::Args&, hipStream_t) {
  return hipErrorInvalidValue;  // the float32 down projection does not split (make_plan)
}
template <>
hipError_t launch_dx_split_kt<float, false>(int, const GemmArgs& ga, const EpiPartial<float>::Args& ea, hipStream_t s) {
  return launch_f32_tile<64, 64, false, true, 1, EpiPartial<float>>(ga, ea, s);
}

template <int BM, int BN, typename Epi>
static hipError_t launch_f32_group(GemmGroup<typename Epi::Args>& grp, hipStream_t s) {
  constexpr auto kern = gemm_f32_group_kernel<BM, BN, Epi>;
  constexpr int LDS = F32Config<BM, BN, true, true, 1>::LDS_BYTES;
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, LDS>, s)) return e;
  int total = 0;
  for (int g = 0; g < grp.count; ++g) {
    grp.first[g] = total;
    total += ((grp.ga[g].M + BM - 1) / BM) * ((grp.ga[g].N + BN - 1) / BN) * (Epi::SPLIT ? grp.ga[g].splits : 1);
  }
  for (int g = grp.count; g <= GEMM_GROUP_MAX; ++g) grp.first[g] = total;
  hipLaunchKernelGGL(kern, dim3(total), dim3(256), LDS, s, grp);
  return hipGetLastError();
}
template <>
hipError_t launch_dw_group<float>(int tc, GemmGroup<EpiStore<float>::Args>& grp, hipStream_t s) {
  if (tc == TILE_F32_128) return launch_f32_group<128, 128, EpiStore<float>>(grp, s);
  if (tc == TILE_F32_64X128) return launch_f32_group<64, 128, EpiStore<float>>(grp, s);
  return launch_f32_group<64, 64, EpiStore<float>>(grp, s);
}
template <>
hipError_t launch_dw_group_split<float>(GemmGroup<EpiPartial<float>::Args>& grp, hipStream_t s) {
  return launch_f32_group<64, 64, EpiPartial<float>>(grp, s);
}

}  // namespace gmlp
