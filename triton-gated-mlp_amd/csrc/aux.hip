// HBM-bound helper kernels: element-wise gating backward, deterministic column sums (bias
// gradients) and the stand-alone dropout keep-mask generator.
#include "launch.hpp"

namespace gmlp {

template <typename T>
__global__ void __launch_bounds__(256)
    gating_bwd_kernel(const T* __restrict__ dh, const T* __restrict__ g, const T* __restrict__ u,
                      T* __restrict__ dg, T* __restrict__ du, size_t n8, int act,
                      DropoutParams d) {
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += stride) {
    size_t e = i * 8;
    float v[8];
    load_w<T, 8>(dh + e, v);
    gating_bwd_w<T, 8>(act, d, e, v, g, u, dg, du);
  }
}

template <typename T>
hipError_t launch_gating_bwd(const T* dh, const T* g, const T* u, T* dg, T* du, int64_t M, int64_t N,
                             int act, const DropoutParams& d, hipStream_t s) {
  size_t n8 = (size_t)M * N / 8;
  if (n8 == 0) return hipSuccess;
  size_t blocks = (n8 + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  hipLaunchKernelGGL(gating_bwd_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, dh, g, u, dg, du,
                     n8, act, d);
  return hipGetLastError();
}
template hipError_t launch_gating_bwd<f16>(const f16*, const f16*, const f16*, f16*, f16*, int64_t,
                                           int64_t, int, const DropoutParams&, hipStream_t);
template hipError_t launch_gating_bwd<bf16>(const bf16*, const bf16*, const bf16*, bf16*, bf16*,
                                            int64_t, int64_t, int, const DropoutParams&,
                                            hipStream_t);
template hipError_t launch_gating_bwd<float>(const float*, const float*, const float*, float*,
                                             float*, int64_t, int64_t, int, const DropoutParams&,
                                             hipStream_t);

// Second stage of a split reduction: adds the partial results up in split order (deterministic)
// and hands 8 consecutive columns of one row to the epilogue the unsplit GEMM would have run.
// Outputs of short batches are a few thousand lanes' work, so the chain of a lane's loads decides: the
// partial sums of 8 splits (4 with two accumulator sets) are in flight together, and small outputs go
// out as workgroups of one wavefront, which spread over more CUs.  M=40, K=4096, N=14336: down
// projection, 14 splits, 6.2 us -> 4.7; M=66,
// K=3208, N=9568: down 6.3 -> 4.2, dX 6.6 -> 4.7.  (All 256 threads wide, the short ones stay at 5; one
// wavefront wide, outputs of 65536 lanes or more gain nothing and large ones lose 1 us of 8.)
template <typename T, typename Epi, int SETS>
__global__ void __launch_bounds__(256)
    splitk_reduce_kernel(const float* __restrict__ ws, int splits, size_t split_stride, size_t acc_stride,
                         typename Epi::Args ea, size_t n8, int N) {
  size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += step) {
    size_t e = i * 8;
    alignas(16) float v[2][8];
#pragma unroll
    for (int r = 0; r < 8; ++r) v[0][r] = v[1][r] = 0.f;
    int s = 0;
    auto add = [&](auto count) __attribute__((always_inline)) {
      constexpr int U = decltype(count)::value;
      f32x4 t[U][SETS][2];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int b = 0; b < SETS; ++b) {
          const float* p = ws + (size_t)(s + u) * split_stride + (b ? acc_stride : 0) + e;
          t[u][b][0] = *(const f32x4*)p;
          t[u][b][1] = *(const f32x4*)(p + 4);
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int b = 0; b < SETS; ++b)
#pragma unroll
          for (int r = 0; r < 8; ++r) v[b][r] += t[u][b][r / 4][r % 4];
      s += U;
    };
    if constexpr (SETS == 1)
      while (s + 8 <= splits) add(std::integral_constant<int, 8>{});
    while (s + 4 <= splits) add(std::integral_constant<int, 4>{});
    if (s + 2 <= splits) add(std::integral_constant<int, 2>{});
    if (s < splits) add(std::integral_constant<int, 1>{});
    Epi::template apply<8>(ea, (int)(e / (size_t)N), (int)(e % (size_t)N), v[0], v[1]);
  }
}

template <typename T, typename Epi>
hipError_t launch_splitk_reduce(const float* ws, int splits, size_t split_stride, size_t acc_stride,
                                const typename Epi::Args& ea, int64_t M, int64_t N, hipStream_t s) {
  constexpr int SETS = std::is_same<Epi, EpiGateUp<T>>::value ? 2 : 1;
  if ((acc_stride != 0) != (SETS == 2)) return hipErrorInvalidValue;
  size_t n8 = (size_t)M * N / 8;
  if (n8 == 0) return hipSuccess;
  const unsigned threads = n8 < 256 * 256 ? 64 : 256;
  size_t blocks = (n8 + threads - 1) / threads;
  if (blocks > 256 * 8) blocks = 256 * 8;
  hipLaunchKernelGGL((splitk_reduce_kernel<T, Epi, SETS>), dim3((unsigned)blocks), dim3(threads), 0, s, ws, splits,
                     split_stride, acc_stride, ea, n8, (int)N);
  return hipGetLastError();
}
#define GMLP_REDUCE_INST(T, EPI)                                                                    \
  template hipError_t launch_splitk_reduce<T, EPI<T>>(const float*, int, size_t, size_t,            \
                                                      const EPI<T>::Args&, int64_t, int64_t, hipStream_t);
GMLP_REDUCE_INST(float, EpiStore)
GMLP_REDUCE_INST(float, EpiGateUp)
GMLP_REDUCE_INST(float, EpiDh)
GMLP_REDUCE_INST(f16, EpiDh)
GMLP_REDUCE_INST(bf16, EpiDh)
GMLP_REDUCE_INST(f16, EpiStore)
GMLP_REDUCE_INST(bf16, EpiStore)
GMLP_REDUCE_INST(f16, EpiGateUp)
GMLP_REDUCE_INST(bf16, EpiGateUp)
#undef GMLP_REDUCE_INST

// The same for the gradients of one pass (contiguous outputs without a bias): blockIdx.y selects the problem.
template <typename T>
__global__ void __launch_bounds__(256) splitk_reduce_group_kernel(ReduceGroup<T> g) {
  const int p = blockIdx.y;
  const float* __restrict__ ws = g.ws[p];
  const size_t n = g.n[p], step = (size_t)gridDim.x * 256 * 8;
  for (size_t e = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8; e < n; e += step) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll 4
    for (int i = 0; i < g.splits[p]; ++i) {
      a += *(const f32x4*)(ws + (size_t)i * n + e);
      b += *(const f32x4*)(ws + (size_t)i * n + e + 4);
    }
    const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    store_w<T, 8, true>(g.out[p] + e, v);
  }
}
template <typename T>
hipError_t launch_splitk_reduce_group(const ReduceGroup<T>& g, hipStream_t s) {
  size_t most = 0;
  for (int i = 0; i < g.count; ++i)
    if (g.n[i] > most) most = g.n[i];
  size_t blocks = (most / 8 + 255) / 256;
  if (blocks > 256 * 8) blocks = 256 * 8;
  hipLaunchKernelGGL(splitk_reduce_group_kernel<T>, dim3((unsigned)blocks, g.count), dim3(256), 0, s, g);
  return hipGetLastError();
}
#define GMLP_REDUCE_GROUP_INST(T) template hipError_t launch_splitk_reduce_group<T>(const ReduceGroup<T>&, hipStream_t);
GMLP_REDUCE_GROUP_INST(f16)
GMLP_REDUCE_GROUP_INST(bf16)
GMLP_REDUCE_GROUP_INST(float)
#undef GMLP_REDUCE_GROUP_INST

// Column sums in a fixed order: COLSUM_SPLITS row ranges, each summed row by row, then the ranges' sums in
// four runs of 16 and the four totals.  Up to COLSUM_GROUP_MAX arrays with the same number of rows share
// the launches (the bias gradients of one backward pass); the grid's last dimension selects the array.
//
// Short batches, one launch: a workgroup does all of it for 64 columns, one range to every 8 threads (8
// columns each), and the ranges' sums change hands through LDS.  Long ones, two: the chain of loads of a
// range grows with the batch, and narrow arrays have too few workgroups; fp32 partial sums in memory.  Both
// add in the same order.  Three arrays of N, N and K columns, bf16, two launches -> one (us): M=32, N=K=32
// 5.2 -> 3.5, M=200, N=704, K=256 5.3 -> 3.5, M=1357, N=3096, K=1160 8.8 -> 8.4, M=2048, N=5632, K=2048
// 13.8 -> 11.8; M=5000, N=600, K=200 9.9 -> 14.3, M=8192, N=8192, K=2048 75 -> 83.  (And one launch less for
// the host, 3 to 4 us of passes that it bounds.)
constexpr int64_t COLSUM_ONE_LAUNCH_MAX_M = 2560;  // 40 rows, five batches of loads, to a range

template <typename T>
__global__ void __launch_bounds__(COLSUM_SPLITS * 8) colsum_kernel(ColsumGroup<T> g, int64_t M) {
  __shared__ __align__(16) char lds[COLSUM_LDS_BYTES];
  const int64_t c0 = (int64_t)blockIdx.x * COLSUM_COLS;
  if (c0 < g.C[blockIdx.y]) colsum_body<T, COLSUM_SPLITS * 8>(g.a[blockIdx.y], g.out[blockIdx.y], g.C[blockIdx.y], c0, M, lds);
}

template <typename T>
__global__ void __launch_bounds__(256) colsum_partial_kernel(ColsumGroup<T> g, int64_t M) {
  const T* __restrict__ a = g.a[blockIdx.z];
  float* __restrict__ ws = g.ws[blockIdx.z];
  const int64_t C = g.C[blockIdx.z];
  int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (c >= C) return;
  int64_t rows = (M + COLSUM_SPLITS - 1) / COLSUM_SPLITS;
  int64_t r0 = blockIdx.y * rows, r1 = r0 + rows < M ? r0 + rows : M;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int64_t r = r0;
  for (; r + 4 <= r1; r += 4) {  // four independent 16-byte loads in flight per lane
    float t[4][8];
#pragma unroll
    for (int u = 0; u < 4; ++u) load_w<T, 8>(a + (r + u) * C + c, t[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 8; ++q) s[q] += t[u][q];
  }
  for (; r < r1; ++r) {
    float t[8];
    load_w<T, 8>(a + r * C + c, t);
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] += t[q];
  }
  float* p = ws + (int64_t)blockIdx.y * C + c;
  *(f32x4*)p = f32x4{s[0], s[1], s[2], s[3]};
  *(f32x4*)(p + 4) = f32x4{s[4], s[5], s[6], s[7]};
}

// Each of a workgroup's four wavefronts adds up 16 of the 64 partial sums, all loads in flight
// together, for the same 64 x 4 columns; the first one adds the four totals.  (One lane walking all 64
// took 7.6 us at three arrays of 5632, 5632 and 2048 columns, this takes 4.8.)
template <typename T>
__global__ void __launch_bounds__(256) colsum_final_kernel(ColsumGroup<T> g) {
  constexpr int WAVES = 4, PER = COLSUM_SPLITS / WAVES;
  __shared__ f32x4 part[WAVES - 1][64];
  const float* __restrict__ ws = g.ws[blockIdx.z];
  const int64_t C = g.C[blockIdx.z];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c = ((int64_t)blockIdx.x * 64 + lane) * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (c < C) {
    f32x4 t[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) t[i] = *(const f32x4*)(ws + (int64_t)(wave * PER + i) * C + c);
#pragma unroll
    for (int i = 0; i < PER; ++i) s += t[i];
  }
  if (wave > 0) part[wave - 1][lane] = s;
  __syncthreads();
  if (wave > 0 || c >= C) return;
#pragma unroll
  for (int w = 0; w < WAVES - 1; ++w) s += part[w][lane];
  float t[4] = {s[0], s[1], s[2], s[3]};
  store_w<T, 4>(g.out[blockIdx.z] + c, t);
}

size_t colsum_workspace_bytes(int64_t, int64_t C) { return (size_t)COLSUM_SPLITS * C * sizeof(float); }

template <typename T>
hipError_t launch_colsum_group(const ColsumGroup<T>& g, int count, int64_t M, hipStream_t s) {
  int64_t cmax = 0;
  for (int i = 0; i < count; ++i) cmax = g.C[i] > cmax ? g.C[i] : cmax;
  if (M <= COLSUM_ONE_LAUNCH_MAX_M) {
    hipLaunchKernelGGL(colsum_kernel<T>, dim3((unsigned)((cmax + COLSUM_COLS - 1) / COLSUM_COLS), count), dim3(COLSUM_SPLITS * 8),
                       0, s, g, M);
    return hipGetLastError();
  }
  unsigned bx8 = (unsigned)((cmax / 8 + 255) / 256), bx4 = (unsigned)((cmax / 4 + 63) / 64);
  hipLaunchKernelGGL(colsum_partial_kernel<T>, dim3(bx8, COLSUM_SPLITS, count), dim3(256), 0, s, g, M);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(colsum_final_kernel<T>, dim3(bx4, 1, count), dim3(256), 0, s, g);
  return hipGetLastError();
}
template hipError_t launch_colsum_group<f16>(const ColsumGroup<f16>&, int, int64_t, hipStream_t);
template hipError_t launch_colsum_group<bf16>(const ColsumGroup<bf16>&, int, int64_t, hipStream_t);
template hipError_t launch_colsum_group<float>(const ColsumGroup<float>&, int, int64_t, hipStream_t);

// Column sums for callers that cannot allocate: the partial sums of the first stage live in this
// array instead of a caller's workspace.  Every GPU the library runs on holds its own copy, at
// its own address, until the process ends (COLSUM_SPLITS x COLSUM_STATIC_MAX_C floats = 8 MiB).
// The name below is a host-side handle, not a device address: host code only ever uses the
// pointer hipGetSymbolAddress returned for the current device.
static __device__ __align__(256) float scratch[(size_t)COLSUM_SPLITS * COLSUM_STATIC_MAX_C];

hipError_t colsum_static_scratch(float** out, hipStream_t s) {
  static std::atomic<float*> known[64];  // per device
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  const bool tracked = dev >= 0 && dev < 64;
  float* p = tracked ? known[dev].load(std::memory_order_acquire) : nullptr;
  if (p == nullptr) {
    // first use on this device (gmlp_init makes it ahead of time): a symbol lookup is not
    // something to do while the stream is being captured
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipError_t e = hipStreamIsCapturing(s, &st)) return e;
    if (st != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
    void* q = nullptr;
    if (hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch))) return e;
    if (q == nullptr) return hipErrorInvalidSymbol;
    p = (float*)q;
    if (tracked) known[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return hipSuccess;
}

// The first stage writes every partial sum the second stage reads (all COLSUM_SPLITS row ranges of
// all C columns, zeros for empty ranges), so nothing in the array has to be cleared between calls.
template <typename T>
hipError_t launch_colsum_static(const T* a, T* out, int64_t M, int64_t C, hipStream_t s) {
  float* ws = nullptr;
  if (hipError_t e = colsum_static_scratch(&ws, s)) return e;
  ColsumGroup<T> g = {};
  g.a[0] = a;
  g.out[0] = out;
  g.ws[0] = ws;
  g.C[0] = C;
  return launch_colsum_group<T>(g, 1, M, s);
}
template hipError_t launch_colsum_static<f16>(const f16*, f16*, int64_t, int64_t, hipStream_t);
template hipError_t launch_colsum_static<bf16>(const bf16*, bf16*, int64_t, int64_t, hipStream_t);
template hipError_t launch_colsum_static<float>(const float*, float*, int64_t, int64_t, hipStream_t);

__global__ void __launch_bounds__(256)
    dropout_mask_kernel(uint8_t* __restrict__ mask, size_t n4, DropoutParams d) {
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
    bool keep[4];
    uint32_t packed = 0x01010101u;
    if (d.enabled) {
      dropout_keep4(d, i, keep);
      packed = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) packed |= (keep[r] ? 1u : 0u) << (8 * r);
    }
    *(uint32_t*)(mask + i * 4) = packed;
  }
}

hipError_t launch_dropout_mask(uint8_t* mask, int64_t M, int64_t N, const DropoutParams& d,
                               hipStream_t s) {
  size_t n4 = (size_t)M * N / 4;
  if (n4 == 0) return hipSuccess;
  size_t blocks = (n4 + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  hipLaunchKernelGGL(dropout_mask_kernel, dim3((unsigned)blocks), dim3(256), 0, s, mask, n4, d);
  return hipGetLastError();
}

}  // namespace gmlp
