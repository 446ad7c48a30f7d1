// float32 path: the GEMMs and fused epilogues for callers that keep the module in float32 (as the
// reference's own tests do), on the bf16 matrix cores: every operand element is split into three bf16
// numbers and a product taken as eight (gemm_f32_split.hpp), which at the matrix cores' nominal rates cost half of the
// time of the fp32 MFMA (v_mfma_f32_32x32x2_f32: 157 TFLOP/s; 2500 bf16).
//
// Precision.  A product enters the sum to 2^-33 of itself.  A bf16 MFMA does not round its sums to nearest (with one
// accumulator a sum of one term comes out up to 2.6 half units off by six products, 1.9 by eight), so the seven products that are at most 2^-8 of the whole go to an accumulator of their own, tile by tile, which
// joins the one of the first parts by an addition.  A sum of one term is then rounded once, as by fp32 MFMAs (largest
// error 1.00 half units, root mean square 0.47, both), and longer ones come out closer, by fewer roundings:
// relative error against float64 at M=2048, K=1024, N=2816, fp32 MFMAs -> one accumulator for six products -> this:
// G 5.7e-7 -> 4.9e-7 -> 2.1e-7, Y 9.5e-7 -> 4.0e-7 -> 1.8e-7, dX 1.34e-6 -> 5.9e-7 -> 2.5e-7, dW 8.1e-7 -> 4.9e-7 ->
// 2.1e-7 (10 shapes of 1 to 6974 rows: sums of one term the same as by fp32 MFMAs, of 32 and more 0.2 to 0.6 of the error).
//
// Bound: the matrix cores at the board's power limit.  M=4096, K=2048, N=5632, fp32 MFMAs -> this (us, TFLOP/s of the
// float32 product): gate/up 1424 -> 1182 (160), down 721 -> 582 (162), dH 772 -> 611 (155), dX 1441 -> 1148 (165),
// weight gradients 2245 -> 1699 (167); 167 is 1334 of bf16.  (Six products in one accumulator: 1027, 498, 516, 960, 1419.)
//
// A tile of 128 x 128 outputs (or 64 x 64) by 32 reduction elements per workgroup of 4 wavefronts.  The
// split is done once per workgroup on the way from global memory to LDS (13 VALU instructions per two
// elements: two or three between two MFMAs), not on every fragment read.  128 x 128: one LDS stage (48 KiB) and all
// of a tile's fragments in registers (96 VGPRs); the next tile is written while the MFMAs of the current
// one run, and a CU holds two workgroups, one of which multiplies while the other waits at a barrier or
// for LDS (128 x 128 x 32 per CU: 1.80 us with one workgroup, 1.44 each with two).  64 x 64 tiles fill the
// chip on small problems, where a launch is as long as its chain of reduction tiles: two LDS stages (one
// barrier a tile) and three reduction tiles in flight in registers (down projection at M=64, K=256, N=1024, one chain:
// 27.8 us with one in flight, 26.0 with three).  Reading the fragments of the next tile ahead as well costs
// the registers of a third workgroup per CU and was 3 to 5 % slower.
#include "gemm_f32_split.hpp"
#include "launch.hpp"

namespace gmlp {

// What the chunks beyond the end of a reduction are fetched from.
static __device__ __align__(16) float f32_zeros[8];

// Which plane of A and which of B the eight products take, smallest first.
constexpr int PRODUCTS = 8;
constexpr int PROD_A[PRODUCTS] = {2, 1, 2, 0, 1, 1, 0, 0};
constexpr int PROD_B[PRODUCTS] = {1, 2, 0, 2, 1, 0, 1, 0};

// Workgroups on a CU, which the registers have to allow.
constexpr int f32_per_cu(int bm, int nb) { return bm == 64 && nb == 1 ? 3 : 2; }

template <int BM, int BN, bool A_KS, bool B_KS, int NB>
struct F32Config {
  static constexpr int BK = 32, NT = 256, WGM = 2, WGN = 2;
  typedef SplitTile<BM, A_KS, NT> AT;
  typedef SplitTile<BN, B_KS, NT> BT;
  static constexpr int WTM = BM / WGM, WTN = BN / WGN, TM = WTM / 16, TN = WTN / 16, G = NB * TN;
  static constexpr int ELD = WTN + 4;
  static constexpr int NS = BM == 64 ? 2 : 1, PF = BM == 64 ? 3 : 1;  // LDS stages; tiles in flight in registers
  static constexpr int STAGE = AT::BYTES + NB * BT::BYTES;
  static constexpr int MAIN_BYTES = NS * STAGE, EPI_BYTES = 4 * NB * 16 * ELD * 4;
  static constexpr int LDS_BYTES = MAIN_BYTES > EPI_BYTES ? MAIN_BYTES : EPI_BYTES;
};

// What the split does not give: operands of magnitude 2^111 and more, infinities among them, leave a NaN
// as their residual, and results of 2^96 and more overflow in the scaled accumulators.  Accumulators that are
// not finite are therefore computed again with fp32 MFMAs; overflows, infinities and NaNs then come out
// as IEEE arithmetic gives them.  A launch with few of them takes up to 1.7 times as long, one in which every output is
// done again two to three times (gate/up of x scaled by 2^100 at M=4096, K=2048, N=5632 1180 -> 3800 us; weight gradients
// with a row of infinities 1700 -> 4420, all on fp32 MFMAs 2220).  Before, each such output was one lane's dot product:
// 49000 and 51000 us.
// 16 rows from m and G times 16 columns (of G / TN operands) from n over reduction tiles [kt_first, kt_end), laid out as
// the accumulators; operands straight from global memory, 32 reduction elements at a time, lane / 16 choosing four of each half.
template <bool A_KS, bool B_KS, int G, int TN>
__device__ __forceinline__ void f32_again(const GemmArgs& ga, f32x4 (&sum)[G], int m, int n, int kt_seg, int kt_first, int kt_end, int lane) {
#pragma unroll
  for (int g = 0; g < G; ++g) sum[g] = f32x4{0.f, 0.f, 0.f, 0.f};
  // (beyond the matrix: its last row or column, which is not stored)
  auto four = [&](auto strided, const float* p, int ld, int row, int k, int end) __attribute__((always_inline)) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (decltype(strided)::value) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j < end) v[j] = p[(size_t)(k + j) * ld + row];
    } else if (k < end) {
      v = *(const f32x4*)(p + (size_t)row * ld + k);
    }
    return v;
  };
  for (int s = 0; s < ga.nseg; ++s) {
    const int k0 = max(kt_first - s * kt_seg, 0) * 32, k1 = min(min(kt_end - s * kt_seg, kt_seg) * 32, ga.K);
    const float* pa = (const float*)ga.A[s];
#pragma unroll 1
    for (int k = k0; k < k1; k += 32) {
      f32x4 a[2], b[2][G];
      const int r = lane & 15;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kl = k + 16 * h + 4 * (lane >> 4);
        a[h] = four(std::integral_constant<bool, A_KS>{}, pa, ga.lda, min(m + r, ga.M - 1), kl, k1);
#pragma unroll
        for (int g = 0; g < G; ++g)
          b[h][g] = four(std::integral_constant<bool, B_KS>{}, (const float*)ga.B[G > TN ? g / TN : s], ga.ldb,
                         min(n + g % TN * 16 + r, ga.N - 1), kl, k1);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int g = 0; g < G; ++g) sum[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[h][g][j], a[h][j], sum[g], 0, 0, 0);
    }
  }
}

// HALVES = 2: a workgroup of twice the wavefronts, whose second half reduces the second half of the range.
template <int BM, int BN, bool A_KS, bool B_KS, int NB, typename Epi, int HALVES = 1>
__device__ __forceinline__ void gemm_f32_body(const GemmArgs& ga, typename Epi::Args ea, int pid, int nwg) {
  typedef F32Config<BM, BN, A_KS, B_KS, NB> Cfg;
  typedef typename Cfg::AT AT;
  typedef typename Cfg::BT BT;
  constexpr int BK = Cfg::BK, TM = Cfg::TM, TN = Cfg::TN, G = Cfg::G, WTM = Cfg::WTM, WTN = Cfg::WTN;
  extern __shared__ __align__(1024) char smem_raw[];

  const int half = HALVES == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  char* const smem = smem_raw + half * Cfg::LDS_BYTES;
  const int tid = threadIdx.x - half * 256, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
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
  if constexpr (HALVES == 2) {  // (as many tiles each, for the barriers; one past the end reads zeros)
    static_assert(!Epi::SPLIT && NB == 1, "built for the down projection");
    const int per = (kt_all + 1) / 2;
    kt_first = half * per;
    kt_end = kt_first + per;
  }

  f32x4 acc[G][TM];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  AT at;
  BT bt[NB];
  constexpr int NS = Cfg::NS, PF = Cfg::PF;
  f32x4 araw[PF][AT::CHUNKS][2], braw[PF][NB][BT::CHUNKS][2];
  int seg = HALVES == 1 && kt_first >= kt_seg ? 1 : 0, kleft = 0;
  auto start = [&](int kk) __attribute__((always_inline)) {
    at.start((const float*)ga.A[seg], ga.lda, m0, kk * BK, ga.M, tid);
#pragma unroll
    for (int b = 0; b < NB; ++b) bt[b].start((const float*)ga.B[NB == 2 ? b : seg], ga.ldb, n0, kk * BK, ga.N, tid);
    kleft = ga.K - kk * BK;
  };
  // On into the second reduction segment.
  auto turn = [&]() __attribute__((always_inline)) {
    if (NB == 1 && kleft <= 0 && seg + 1 < ga.nseg) {
      seg = 1;
      start(0);
    }
  };
  constexpr int CH = AT::CHUNKS + NB * BT::CHUNKS;
  auto load_chunk = [&](int p, int c) __attribute__((always_inline)) {
    if (c < AT::CHUNKS) {
      at.load1(araw[p][c], c, ga.lda, kleft, f32_zeros);
    } else {
      const int b = (c - AT::CHUNKS) / BT::CHUNKS, i = (c - AT::CHUNKS) % BT::CHUNKS;
      bt[b].load1(braw[p][b][i], i, ga.ldb, kleft, f32_zeros);
    }
  };
  auto store_chunk = [&](int p, int c, char* st) __attribute__((always_inline)) {
    if (c < AT::CHUNKS) {
      AT::store(st, araw[p][c], c, tid);
    } else {
      const int b = (c - AT::CHUNKS) / BT::CHUNKS, i = (c - AT::CHUNKS) % BT::CHUNKS;
      BT::store(st + AT::BYTES + b * BT::BYTES, braw[p][b][i], i, tid);
    }
  };

  start(kt_first - seg * kt_seg);
#pragma unroll
  for (int p = 0; p < PF; ++p) {
#pragma unroll
    for (int c = 0; c < CH; ++c) load_chunk(p, c);
    kleft -= BK;
    turn();
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    store_chunk(0, c, smem);
    load_chunk(0, c);
  }
  kleft -= BK;

  // Reduction tile t of the range, which is in LDS; tile t + 1, in registers (slot p), goes there meanwhile.
  auto tile = [&](int t, int p) __attribute__((always_inline)) {
    const char* cur = smem + (NS == 2 ? (t & 1) * Cfg::STAGE : 0);
    char* nxt = smem + (NS == 2 ? ((t + 1) & 1) * Cfg::STAGE : 0);
    turn();
    __syncthreads();  // the tile is in LDS
    bf16x8 af[3][TM], bf[3][G];
#pragma unroll
    for (int s = 2; s >= 0; --s) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[s][i] = AT::frag(cur, s, wm * WTM + i * 16, lane);
#pragma unroll
      for (int g = 0; g < G; ++g)
        bf[s][g] = BT::frag(cur + AT::BYTES + (g / TN) * BT::BYTES, s, wn * WTN + (g % TN) * 16, lane);
    }
    if (NS == 1) __syncthreads();  // and every wavefront has its part of it in registers
    __builtin_amdgcn_sched_barrier(0);
    // Four 16 x 16 outputs at a time, the small products of the tile in accumulators of their own.
    constexpr int TOGETHER = 4, GROUPS = TM * G / TOGETHER;
    static_assert(TM * G % TOGETHER == 0, "whole groups");
#pragma unroll
    for (int f = 0; f < GROUPS; ++f) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (c * GROUPS / CH == f) store_chunk(p, c, nxt), load_chunk(p, c);
      f32x4 small[TOGETHER];
#pragma unroll
      for (int q = 0; q < PRODUCTS; ++q)
#pragma unroll
        for (int e = 0; e < TOGETHER; ++e) {
          const int g = (f * TOGETHER + e) / TM, i = (f * TOGETHER + e) % TM;
          f32x4& sum = q + 1 < PRODUCTS ? small[e] : acc[g][i];
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          // operands swapped: a lane ends up with 4 consecutive output columns of one row
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[PROD_B[q]][g], af[PROD_A[q]][i], q == 0 ? zero : sum, 0, 0, 0);
        }
#pragma unroll
      for (int e = 0; e < TOGETHER; ++e) acc[(f * TOGETHER + e) / TM][(f * TOGETHER + e) % TM] += small[e];
#pragma unroll
      for (int r = 0; r < PRODUCTS * TOGETHER; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // MFMA
        // VALU, as many as there are to an MFMA (splitting, addresses, the sums above): gate/up at M=2048, K=1024, N=2816
        // 204 us with 4 of them on 128-row tiles, 189 with 2, 197 with 1
        __builtin_amdgcn_sched_group_barrier(0x2, BM == 128 ? 2 : 4, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    kleft -= BK;
  };
  // (whole groups of PF tiles first: a branch between two tiles of the loop would have the compiler wait
  // for loads of tiles that are not due yet)
  const int tiles = kt_end - kt_first;
  int t = 0;
  for (; t + PF <= tiles; t += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) tile(t + u, (u + 1) % PF);
  }
#pragma unroll
  for (int u = 0; u + 1 < PF; ++u) {
    if (t + u >= tiles) break;
    tile(t + u, (u + 1) % PF);
  }

#pragma unroll
  for (int i = 0; i < TM; ++i) {
    float not_finite = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        not_finite = fmaf(acc[g][i][r], 0.f, not_finite);
        acc[g][i][r] *= 1.0f / (SPLIT_SCALE * SPLIT_SCALE);
      }
    if (__builtin_amdgcn_ballot_w64(!(not_finite == 0.f)) == 0) continue;
    f32x4 again[G];
    f32_again<A_KS, B_KS, G, TN>(ga, again, m0 + wm * WTM + i * 16, n0 + wn * WTN, kt_seg, kt_first, kt_end, lane);
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!(acc[g][i][r] * 0.f == 0.f)) acc[g][i][r] = again[g][r];
  }

  __syncthreads();  // the slabs overwrite the operand tiles
  if constexpr (HALVES == 2) {  // the second half's sums change hands through its part of LDS
    f32x4* const other = (f32x4*)(smem_raw + Cfg::LDS_BYTES) + tid;
    static_assert(G * TM * 256 * 16 <= Cfg::LDS_BYTES, "accumulators fit");
    if (half == 1) {
#pragma unroll
      for (int q = 0; q < G * TM; ++q) other[q * 256] = acc[q / TM][q % TM];
    }
    __syncthreads();
    if (half == 1) return;
#pragma unroll
    for (int q = 0; q < G * TM; ++q) acc[q / TM][q % TM] += other[q * 256];
  }
  constexpr int ELD = Cfg::ELD, CPW = WTN / 4, ITEMS = 16 * CPW / 64;
  static_assert(16 * CPW % 64 == 0, "slab items divide over the lanes");
  float* slab = (float*)smem + wave * NB * 16 * ELD;
  const int mrow = lane & 15, nsub = 4 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int mw = m0 + wm * WTM + i * 16, nw = n0 + wn * WTN;
    typename Epi::template Prefetch<4> pf[ITEMS];
    if (Epi::PREFETCH_DEPTH > 0) {
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {  // beyond the edge: the last valid elements, dropped below
        const int q = it * 64 + lane;
        Epi::template prefetch<4>(ea, min(mw + q / CPW, ga.M - 1), min(nw + q % CPW * 4, ga.N - 4), pf[it]);
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
      *(f32x4*)(slab + ((g / TN) * 16 + mrow) * ELD + (g % TN) * 16 + nsub) = acc[g][i];
    // (same-wavefront LDS writes and reads are ordered)
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int q = it * 64 + lane, row = q / CPW, col = q % CPW * 4, m = mw + row, n = nw + col;
      alignas(16) float v0[4], v1[4];
      *(f32x4*)v0 = *(const f32x4*)(slab + row * ELD + col);
      *(f32x4*)v1 = *(const f32x4*)(slab + ((NB - 1) * 16 + row) * ELD + col);
      if (m < ga.M && n < ga.N) Epi::template apply<4, ACT_RUNTIME>(ea, m, n, v0, v1, pf[it]);
    }
  }
}

template <int BM, int BN, bool A_KS, bool B_KS, int NB, typename Epi>
__global__ void __launch_bounds__(256, f32_per_cu(BM, NB)) gemm_f32_kernel(GemmArgs ga, typename Epi::Args ea) {
  gemm_f32_body<BM, BN, A_KS, B_KS, NB, Epi>(ga, ea, blockIdx.x, gridDim.x);
}

// Both halves of the reduction by one workgroup, for down projections of at most one workgroup per CU that leave no partial
// sums in memory: the launch is as long as its chain of reduction tiles, and a CU has room for two chains.  fp32 MFMAs ->
// six products, one chain -> eight, two chains (us): M=1 to 64, K=1024, N=2816 56 -> 66 -> 50, M=64, K=256, N=1024
// 22 -> 26 -> 21, M=8, K=4096, N=11008 209 -> 247 -> 180.  (Gate/up, two accumulator sets: 13.6 -> 12.7 at 8 reduction tiles,
// nothing at M=8, K=4096, N=11008, so it has no such kernel.)
__global__ void __launch_bounds__(512, 2) gemm_f32_halves_kernel(GemmArgs ga, EpiStore<float>::Args ea) {
  gemm_f32_body<64, 64, false, false, 1, EpiStore<float>, 2>(ga, ea, blockIdx.x, gridDim.x);
}

template <int BM, int BN, typename Epi>
__global__ void __launch_bounds__(256, f32_per_cu(BM, 1)) gemm_f32_group_kernel(GemmGroup<typename Epi::Args> grp) {
  int g = 0;
#pragma unroll
  for (int i = 1; i < GEMM_GROUP_MAX; ++i)
    if (i < grp.count && (int)blockIdx.x >= grp.first[i]) g = i;
  gemm_f32_body<BM, BN, true, true, 1, Epi>(grp.ga[g], grp.ea[g], (int)blockIdx.x - grp.first[g],
                                           grp.first[g + 1] - grp.first[g]);
}

// The input gradient, the weight gradients and the bias gradients as one grid (see gemm_pipelined.hpp's of 16-bit
// types), all on square tiles of the same size.  Backward passes, launches of their own -> one grid: 512x512x512 42 -> 34 us,
// 684x56x224 27 -> 20 and with biases 32 -> 20, 1280x320x1216 88 -> 79 and 92 -> 77.
template <int B, typename EpiX, typename EpiW>
__global__ void __launch_bounds__(256, f32_per_cu(B, 1)) gemm_f32_dx_dw_kernel(DxDwGroup<float, EpiX, EpiW> grp) {
  int pid = (int)blockIdx.x;
  if (grp.nsums > 0 && pid >= grp.sum_first[0]) {
    extern __shared__ __align__(1024) char smem[];
    int i = 0;
#pragma unroll
    for (int k = 1; k < COLSUM_GROUP_MAX; ++k)
      if (k < grp.nsums && pid >= grp.sum_first[k]) i = k;
    colsum_body<float, 256>(grp.sums.a[i], grp.sums.out[i], grp.sums.C[i], (int64_t)(pid - grp.sum_first[i]) * COLSUM_COLS,
                            grp.sum_rows, smem);
    return;
  }
  if (pid >= grp.x0 && pid < grp.x0 + grp.dx_wgs) {
    gemm_f32_body<B, B, false, true, 1, EpiX>(grp.gx, grp.ex, pid - grp.x0, grp.dx_wgs);
    return;
  }
  if (pid >= grp.x0 + grp.dx_wgs) pid -= grp.dx_wgs;
  int g = 0;
#pragma unroll
  for (int i = 1; i < GEMM_GROUP_MAX; ++i)
    if (i < grp.w.count && pid >= grp.w.first[i]) g = i;
  gemm_f32_body<B, B, true, true, 1, EpiW>(grp.w.ga[g], grp.w.ea[g], pid - grp.w.first[g], grp.w.first[g + 1] - grp.w.first[g]);
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
// One accumulator set: 128x128 or 64x64 tiles; two: 128x64 or 64x64 (x 2).
template <bool A_KS, bool B_KS, int NB, typename Epi>
static hipError_t launch_f32(int tile_class, const GemmArgs& ga, const typename Epi::Args& ea, hipStream_t s) {
  if (tile_class == TILE_F32_128) return launch_f32_tile<128, 128 / NB, A_KS, B_KS, NB, Epi>(ga, ea, s);
  return launch_f32_tile<64, 64, A_KS, B_KS, NB, Epi>(ga, ea, s);
}

template <>
hipError_t launch_gateup_kt<float, false>(int tc, const GemmArgs& ga, const EpiGateUp<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, false, 2, EpiGateUp<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_linear_kt<float, false>(int tc, const GemmArgs& ga, const EpiStore<float>::Args& ea, hipStream_t s) {
  if (tc != TILE_F32_HALVES) return launch_f32<false, false, 1, EpiStore<float>>(tc, ga, ea, s);
  constexpr auto kern = gemm_f32_halves_kernel;
  constexpr int LDS = 2 * F32Config<64, 64, false, false, 1>::LDS_BYTES;
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, LDS>, s)) return e;
  hipLaunchKernelGGL(kern, dim3(((ga.M + 63) / 64) * ((ga.N + 63) / 64)), dim3(512), LDS, s, ga, ea);
  return hipGetLastError();
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
template <>
hipError_t launch_gateup_split_kt<float, false>(int tc, const GemmArgs& ga, const EpiPartial<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, false, 2, EpiPartial<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_linear_split_kt<float, false>(int tc, const GemmArgs& ga, const EpiPartial<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, false, 1, EpiPartial<float>>(tc, ga, ea, s);
}
template <>
hipError_t launch_dx_split_kt<float, false>(int tc, const GemmArgs& ga, const EpiPartial<float>::Args& ea, hipStream_t s) {
  return launch_f32<false, true, 1, EpiPartial<float>>(tc, ga, ea, s);
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
  return launch_f32_group<64, 64, EpiStore<float>>(grp, s);
}
template <>
hipError_t launch_dw_group_split<float>(int tc, GemmGroup<EpiPartial<float>::Args>& grp, hipStream_t s) {
  if (tc == TILE_F32_128) return launch_f32_group<128, 128, EpiPartial<float>>(grp, s);
  return launch_f32_group<64, 64, EpiPartial<float>>(grp, s);
}

template <int B, typename EpiX, typename EpiW>
static hipError_t launch_f32_dx_dw(DxDwGroup<float, EpiX, EpiW>& grp, bool dx_first, hipStream_t s) {
  constexpr auto kern = gemm_f32_dx_dw_kernel<B, EpiX, EpiW>;
  constexpr int LDS_X = F32Config<B, B, false, true, 1>::LDS_BYTES, LDS_W = F32Config<B, B, true, true, 1>::LDS_BYTES;
  constexpr int LDS = LDS_X > LDS_W ? LDS_X : LDS_W;
  static_assert(LDS >= COLSUM_LDS_BYTES, "the sums' workgroups use the same allocation");
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, LDS>, s)) return e;
  hipLaunchKernelGGL(kern, dim3(place_dx_dw<B, B, B>(grp, dx_first)), dim3(256), LDS, s, grp);
  return hipGetLastError();
}
template <>
hipError_t launch_dx_dw_kt<float, false>(int tc, DxDwGroup<float, EpiStore<float>>& grp, bool dx_first, hipStream_t s) {
  return tc == TILE_F32_128 ? launch_f32_dx_dw<128>(grp, dx_first, s) : launch_f32_dx_dw<64>(grp, dx_first, s);
}
template <>
hipError_t launch_dx_dw_kt<float, false>(int tc, DxDwGroup<float, EpiPartial<float>>& grp, bool dx_first, hipStream_t s) {
  return tc == TILE_F32_128 ? launch_f32_dx_dw<128>(grp, dx_first, s) : launch_f32_dx_dw<64>(grp, dx_first, s);
}
template <>
hipError_t launch_dx_dw_kt<float, false>(int tc, DxDwGroup<float, EpiStore<float>, EpiPartial<float>>& grp, bool dx_first, hipStream_t s) {
  return tc == TILE_F32_128 ? launch_f32_dx_dw<128>(grp, dx_first, s) : launch_f32_dx_dw<64>(grp, dx_first, s);
}
template <>
hipError_t launch_dx_dw_kt<float, false>(int tc, DxDwGroup<float, EpiPartial<float>, EpiPartial<float>>& grp, bool dx_first, hipStream_t s) {
  return tc == TILE_F32_128 ? launch_f32_dx_dw<128>(grp, dx_first, s) : launch_f32_dx_dw<64>(grp, dx_first, s);
}

}  // namespace gmlp
