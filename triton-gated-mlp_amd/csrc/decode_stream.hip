// Skinny-M (M <= 32) forward in two launches, gate/up and down, on the streaming body of decode_stream.hpp.
//
// Which block (chosen in launch_decode_stream; kernel times, us, fp16): the height decides what a block
// costs in token operands and how well it fits a CU's share of the rows; the row segment of a stage (SEGB)
// how evenly the chunks divide over the wavefronts (16 chunks of 256 elements at K = 4096: 6, 5 and 5; 64 of
// 64: 22, 21 and 21), how soon the first MFMA can start, and how finely the ring's slots take up what the
// loads in flight leave.  512- -> 128-byte segments, W_gate / W_up, 16 rows a block: K=2048, N=8192 M=8
// 17.4 -> 14.6, M=16 19.1 -> 15.4; K=1024, N=4096 9.3 -> 7.1, 10.1 -> 7.6.  Bytes in flight do not decide at
// 96 KiB per CU: four, six and eight wavefronts with 128 to 144 KiB were no faster on any of eleven
// widths.
#include "decode_stream.hpp"

namespace gmlp {

constexpr int DS_WIDE_SEGMENT_MAX_M = 20;     // see ds_tall_gated, ds_short_segments

template <typename T, bool GATED, int HALVES, int MT, int SEGB, int DS_RD, bool TAIL, int RR, int NW>
__global__ void __launch_bounds__(NW * 64) decode_stream_kernel(StreamArgs a) {
  extern __shared__ __align__(1024) char smem[];
  StreamBody<T, GATED, HALVES, MT, SEGB, DS_RD, TAIL, RR, NW> body;
  body.start(a, smem, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), (int)blockIdx.x, (int)gridDim.x);
#pragma unroll
  for (int p = 0; p < DS_RD; ++p) body.issue_stage(a, p, p);
  body.run(a);
  wait_vmem<0>();
}

template <typename T, bool GATED, int HALVES, int MT, int SEGB, int RD, bool TAIL, int RR, int NW>
static hipError_t launch_stream_tail(const StreamArgs& a, int num_cu, hipStream_t s) {
  constexpr int LDS = StreamBody<T, GATED, HALVES, MT, SEGB, RD, TAIL, RR, NW>::LDS_BYTES;
  constexpr auto kern = decode_stream_kernel<T, GATED, HALVES, MT, SEGB, RD, TAIL, RR, NW>;
  if (hipError_t e = allow_dynamic_lds(lds_kernel_of<kern, LDS>, s)) return e;
  hipLaunchKernelGGL(kern, dim3(ds_grid(a.R, num_cu)), dim3(NW * 64), LDS, s, a);
  return hipGetLastError();
}
template <typename T, bool GATED, int HALVES, int MT, int SEGB, int RD, int RR = 16, int NW = 3>
static hipError_t launch_stream(const StreamArgs& a, int num_cu, hipStream_t s) {
  if constexpr (SEGB > 128)  // (rows of whole 128-byte lines are a multiple of 64 elements)
    if (a.red % (SEGB / 2) != 0) return launch_stream_tail<T, GATED, HALVES, MT, SEGB, RD, true, RR, NW>(a, num_cu, s);
  return launch_stream_tail<T, GATED, HALVES, MT, SEGB, RD, false, RR, NW>(a, num_cu, s);
}

bool decode_stream_supported(int M, int K, int N) {
  return M >= 1 && M <= 32 && K % 8 == 0 && N % 8 == 0 && K >= DS_MIN_RED && N >= DS_MIN_RED &&
         (int64_t)K * N * 2 < ((int64_t)1 << 31);
}

// Segments of 128 bytes: reduction lengths that are a multiple of 256 and rows that are one of 64, the
// widths that models have and that this was measured on.  (Never rows that do not start on a 128-byte
// line: every segment touches one line more than it fills, see ds_tall_gated.)  Long segments stream a few
// per cent faster from HBM once a kernel runs long enough for that to count and the token operands cost
// little.  One token tile, whole forward, long -> short: K=1024, N=4096 M=1 14.8 -> 13.8, M=8 16.2 -> 14.0;
// K=4096, N=14336 61.7 -> 61.7, 63.3 -> 59.5; K=6144, N=16384 99.5 -> 101.9, 97.3 -> 97.9; K=2048, N=8192
// 26.9 -> 27.6, 29.6 -> 28.3.  Two: K=8192, N=28672 M=17 230 -> 232, M=32 243 -> 234.
static bool ds_short_segments(int M, int rows, int red) {
  if (red % 256 != 0 || rows % 64 != 0) return false;
  const int64_t elements = (int64_t)rows * red;
  if (M > 16) return M > DS_WIDE_SEGMENT_MAX_M || elements <= ((int64_t)128 << 20);
  return elements <= ((int64_t)(M <= 4 ? 12 : 64) << 20);
}

// Height of a block of W_gate and W_up rows, in units of 16, for segments of 128 bytes: the one whose blocks
// cost a CU's share least, a block costing its rows (the partly empty last one all of them: its missing rows
// leave slots of the ring unused) and its token operands (0.2 of a row of weights per token with two token
// tiles; 0.05 with one).  One tile: 16 or 32 rows (N = 13824, K = 5120, 54 rows per CU, M = 8 47.8 / 46.6;
// N = 11008, K = 4096, 43 rows 30.1 / 33.0), two: up to 80.  M = 32, rows per CU, us at 16 / 32 / 48 / 64 / 80: N = 11008,
// K = 4096, 43 rows 41 / 40 / 34 / 34 / 36; N = 14336, 56 rows 51 / 44 / 51 / 41 / 42; N = 28672, K = 8192,
// 112 rows 179 / 158 / 172 / 150 / 162; N = 18944, K = 3584, 74 rows 65 / 59 / 53 / 61 / 52.  Over 25
// widths and M = 17, 24, 32 the kernel takes 0.89 of the time of the blocks of 16 rows of 256 elements or 32 of 128
// that it took before, M = 6, 10, 16 0.92.
static int ds_gated_height(int M, int N, int num_cu) {
  const bool two = M > 16;
  int best = 1;
  double least = 1e30;
  for (int h = 1; h <= (two ? 5 : 2); ++h) {
    const int rows = 16 * h, full = N / rows / num_cu, rest = N - full * num_cu * rows;
    const int blocks = full + (rest + num_cu * rows - 1) / (num_cu * rows);
    const double cost = blocks * (rows + (two ? 0.2 : 0.05) * M);
    if (cost < least) least = cost, best = h;
  }
  return best;
}

// The other widths.  Blocks of 32 rows of W_gate and W_up, 128 elements a stage (two stages' worth of 16-row
// blocks of 256 elements): half the token operands per weight byte.  With one token tile or little more
// the operands cost less than a block that a CU's share does not fill, so they are taken there only
// where the share rounded up to 16 and to 32 rows is the same, and up to 10 tokens not at all (M=5, K=3840,
// N=6656 33.0 / 32.3).  Rows that do not start on a 128-byte line take the long segments throughout: a
// 256-byte one touches three lines instead of two (K=6712, N=24104, M=1 210 -> 188 us; K=3592, N=8200,
// M=24 61 -> 56; M=32, K=3112, N=7000 is the one that loses, 46.4 -> 47.6).
static bool ds_whole_lines(int red) { return red % 64 == 0; }
static bool ds_tall_gated(int M, int K, int N, int num_cu) {
  if (!ds_whole_lines(K)) return false;
  const int rows = (N + num_cu - 1) / num_cu;
  return M > DS_WIDE_SEGMENT_MAX_M || (M > DS_H_TILED_MIN_M && (rows + 15) / 16 % 2 == 0);
}

template <typename T>
hipError_t launch_decode_stream(const T* x, const T* wg, const T* wu, const T* wd, const T* bg,
                                const T* bu, const T* bd, T* h, T* y, int M, int K, int N,
                                int act, hipStream_t s) {
  int dev = 0, num_cu = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  if (hipError_t e = hipDeviceGetAttribute(&num_cu, hipDeviceAttributeMultiprocessorCount, dev)) return e;
  if (num_cu <= 0) num_cu = 256;
  const int tiled = ds_h_tiled(M);
  StreamArgs a1 = {x, {wg, wu}, {bg, bu}, h, M, N, K, K, N, act, tiled};
  StreamArgs a2 = {h, {wd, wd}, {bd, bd}, y, M, K, N, N, K, ACT_IDENTITY, tiled};
  // Ring depths: what 160 KiB hold (and, two token tiles, what the operands in flight leave in the VGPRs).
  auto gated = [&]() -> hipError_t {
    if (!ds_short_segments(M, N, K) || N < 8 * num_cu) {
      const bool tall = ds_tall_gated(M, K, N, num_cu);
      if (M <= 16) return tall ? launch_stream<T, true, 2, 1, 256, 3>(a1, num_cu, s) : launch_stream<T, true, 1, 1, 512, 3>(a1, num_cu, s);
      return tall ? launch_stream<T, true, 2, 2, 256, 3>(a1, num_cu, s) : launch_stream<T, true, 1, 2, 512, 3>(a1, num_cu, s);
    }
    const int height = ds_gated_height(M, N, num_cu);
    if (M <= 16) return height == 1 ? launch_stream<T, true, 1, 1, 128, 8>(a1, num_cu, s) : launch_stream<T, true, 2, 1, 128, 6>(a1, num_cu, s);
    switch (height) {
      case 1: return launch_stream<T, true, 1, 2, 128, 8>(a1, num_cu, s);
      case 2: return launch_stream<T, true, 2, 2, 128, 6>(a1, num_cu, s);
      case 3: return launch_stream<T, true, 3, 2, 128, 3>(a1, num_cu, s);
      case 4: return launch_stream<T, true, 4, 2, 128, 2>(a1, num_cu, s);
      default: return launch_stream<T, true, 5, 2, 128, 2>(a1, num_cu, s);
    }
  };
  if (hipError_t e = gated()) return e;
  // W_down: 32 rows a block once a CU's share exceeds 16 rows, 16 up to there.  One token tile: segments of
  // 128 bytes, eight stages deep (against 512 / 256 bytes, M = 6 to 16, 25 widths: 0.91 of the time);
  // otherwise 256 elements a stage up to 16 rows and on misaligned rows, 128 beyond (K=6712,
  // N=24104, M=1, 256 elements for 128 188 -> 178 us).  Two tiles: H's operands are as many bytes as the
  // weights, and shorter stages only add instructions (K=2048, N=8192, M=24 128- against 512-byte segments
  // 16.0 / 14.9), so 256 elements up to 16 rows, 128 beyond, and 64 rows at a time from 48 rows (K=16384,
  // N=53248, M=18 807 -> 783 us for the whole forward).
  // Shares of 8 rows or fewer (a CU's loads in flight, not the bytes, bound these): regions of 8 rows, so that every
  // byte of the rings' slots is in flight for a weight, and four wavefronts where the segments are short.  Kernel alone,
  // M=1: K=1024, N=4096 7.8 -> 6.2, K=2048, N=5632 9.5 -> 7.8, K=2048, N=8192 12.0 -> 9.7; M=16 9.5 -> 8.8 and 12.2 ->
  // 10.6; M=24 11.4 -> 10.7 and 13.7 -> 12.9.  Four wavefronts also for whole regions that a share leaves partly
  // empty (M=1: K=2560, N=6912 11.2 -> 9.5, K=3072, N=8192 12.3 -> 10.8; from 14 rows of 16 on equal or 2 % slower).
  // Long segments, one token tile: three slots.  A wavefront has a few stages only, and the ones past the end cost
  // their instructions: whole forwards (launches in a graph, K = 768 to 2048, every kind of row) take 0.92 of the time with
  // six slots up to N = 4096, 0.96 around 8192, 0.97 beyond 12288 (two slots: 0.90, 0.95, 0.99), and 0.92 of the time
  // with regions of 16 rows throughout.  M=1, K=2048, N=8192: 16 rows 23.4, six slots 22.5, three 21.8.  Two token tiles: 8
  // rows take 0.98 of 16.
  const bool half = K <= 8 * num_cu;
  const bool one = K <= 16 * num_cu, lines = ds_whole_lines(N), four = K > 48 * num_cu && lines;
  if (M <= 16) {
    if (ds_short_segments(M, K, N))
      return half                ? launch_stream<T, false, 1, 1, 128, 8, 8, 4>(a2, num_cu, s)
             : K <= 13 * num_cu ? launch_stream<T, false, 1, 1, 128, 8, 16, 4>(a2, num_cu, s)
             : one              ? launch_stream<T, false, 1, 1, 128, 8>(a2, num_cu, s)
                                : launch_stream<T, false, 2, 1, 128, 8>(a2, num_cu, s);
    if (half) return launch_stream<T, false, 1, 1, 512, 3, 8>(a2, num_cu, s);
    if (one) return launch_stream<T, false, 1, 1, 512, 4>(a2, num_cu, s);
    return lines ? launch_stream<T, false, 2, 1, 256, 4>(a2, num_cu, s) : launch_stream<T, false, 2, 1, 512, 3>(a2, num_cu, s);
  }
  if (half) return launch_stream<T, false, 1, 2, 512, 3, 8>(a2, num_cu, s);
  if (four) return launch_stream<T, false, 4, 2, 256, 3>(a2, num_cu, s);
  if (one) return launch_stream<T, false, 1, 2, 512, 3>(a2, num_cu, s);
  return lines ? launch_stream<T, false, 2, 2, 256, 4>(a2, num_cu, s) : launch_stream<T, false, 2, 2, 512, 3>(a2, num_cu, s);
}

template hipError_t launch_decode_stream<f16>(const f16*, const f16*, const f16*, const f16*,
                                              const f16*, const f16*, const f16*, f16*, f16*, int,
                                              int, int, int, hipStream_t);
template hipError_t launch_decode_stream<bf16>(const bf16*, const bf16*, const bf16*, const bf16*,
                                               const bf16*, const bf16*, const bf16*, bf16*, bf16*,
                                               int, int, int, int, hipStream_t);

}  // namespace gmlp
