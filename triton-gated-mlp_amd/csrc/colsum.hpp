// Column sums of 64 columns by one workgroup: the whole of a launch of its own (aux.hip) or some of the
// workgroups of a backward pass's grid (gemm_pipelined.hpp).
#pragma once
#include "gemm.hpp"

namespace gmlp {

constexpr int COLSUM_GROUP_MAX = 3;
template <typename T>
struct ColsumGroup {
  const T* a[COLSUM_GROUP_MAX];   // [M, C[i]]
  T* out[COLSUM_GROUP_MAX];       // [C[i]]
  float* ws[COLSUM_GROUP_MAX];    // colsum_workspace_bytes(M, C[i]) bytes each
  int64_t C[COLSUM_GROUP_MAX];
};

// Row ranges, and columns of a workgroup.
constexpr int COLSUM_SPLITS = 64, COLSUM_COLS = 64;
constexpr int COLSUM_LDS_BYTES = COLSUM_SPLITS * (COLSUM_COLS + 4) * 4;

// Each of the COLSUM_SPLITS row ranges summed row by row, 8 threads to a range (8 columns each), then the ranges'
// sums, which change hands through LDS, in four runs of 16 and the four totals.  With fewer than 8 threads a range
// a thread walks several ranges side by side (as many loads in flight for a workgroup of half the threads).
template <typename T, int THREADS>
__device__ __forceinline__ void colsum_body(const T* __restrict__ a, T* __restrict__ out, int64_t C, int64_t c0, int64_t M, char* lds) {
  constexpr int RUNS = 4, PER = COLSUM_SPLITS / RUNS, AT_ONCE = THREADS / 8, EACH = COLSUM_SPLITS / AT_ONCE;
  static_assert(EACH * AT_ONCE == COLSUM_SPLITS && THREADS >= 64, "whole ranges");
  float (*part)[COLSUM_COLS + 4] = (float (*)[COLSUM_COLS + 4])lds;
  const int range = threadIdx.x / 8, col = threadIdx.x % 8 * 8;
  const int64_t rows = (M + COLSUM_SPLITS - 1) / COLSUM_SPLITS;
  float s[EACH][8] = {};
  if (c0 + col < C) {
    const T* p = a + range * rows * C + c0 + col;
    const int64_t apart = AT_ONCE * rows * C;
    int64_t left[EACH];  // rows of each range, not increasing
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int64_t behind = M - (range + i * AT_ONCE) * rows;
      left[i] = behind < rows ? (behind > 0 ? behind : 0) : rows;
    }
    auto add = [&](auto ranges, auto count, int64_t r) __attribute__((always_inline)) {  // independent loads in flight
      constexpr int N = decltype(ranges)::value, U = decltype(count)::value;
      typename Traits<T>::vec8 t[N][U];
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u) t[i][u] = *(const typename Traits<T>::vec8*)(p + i * apart + (r + u) * C);
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int q = 0; q < 8; ++q) s[i][q] += Traits<T>::to_f32(t[i][u][q]);
    };
    int64_t r = 0;
    auto walk = [&](auto ranges) __attribute__((always_inline)) {
      const int64_t end = left[decltype(ranges)::value - 1];
      for (; r + 8 <= end; r += 8) add(ranges, std::integral_constant<int, 8>{}, r);
      if (r + 4 <= end) { add(ranges, std::integral_constant<int, 4>{}, r); r += 4; }
      if (r + 2 <= end) { add(ranges, std::integral_constant<int, 2>{}, r); r += 2; }
      if (r < end) { add(ranges, std::integral_constant<int, 1>{}, r); r += 1; }
    };
    static_assert(EACH <= 2, "walked side by side, then the first one's last rows");
    walk(std::integral_constant<int, EACH>{});
    if constexpr (EACH == 2) walk(std::integral_constant<int, 1>{});
  }
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    *(f32x4*)&part[range + i * AT_ONCE][col] = f32x4{s[i][0], s[i][1], s[i][2], s[i][3]};
    *(f32x4*)&part[range + i * AT_ONCE][col + 4] = f32x4{s[i][4], s[i][5], s[i][6], s[i][7]};
  }
  __syncthreads();
  // the first wavefront: 16 lanes to a run, 4 columns each
  const int run = threadIdx.x / 16, c = threadIdx.x % 16 * 4;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (run < RUNS) {
#pragma unroll
    for (int i = 0; i < PER; ++i) v += *(const f32x4*)&part[run * PER + i][c];
  }
  __syncthreads();
  if (run < RUNS) *(f32x4*)&part[run][c] = v;
  __syncthreads();
  if (run > 0 || c0 + c >= C) return;
#pragma unroll
  for (int i = 1; i < RUNS; ++i) v += *(const f32x4*)&part[i][c];
  const float t[4] = {v[0], v[1], v[2], v[3]};
  store_w<T, 4>(out + c0 + c, t);
}

}  // namespace gmlp
