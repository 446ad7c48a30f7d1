// float32 GEMM on the bf16 matrix cores: C[M,N] = sum_s sum_k A_s[m,k] * B_s[n,k] with every float32
// operand element, times 2^16, written as the sum of three bf16 numbers, 2^16 x = h + m + l, and the product
// of two of them as the eight products hh, hm, mh, hl, lh, mm, ml, lm, each exact in float32.  Three times 8
// significant bits hold the 24 of a float32, and the factor puts the smallest float32 (2^-149) at the
// smallest bf16 (2^-133; the matrix cores take subnormal ones), so the sum is x exactly for every |x| below
// 2^111.  What is left out of a product, ll, is at most 2^-34 of it: |m| <= 2^-8 |x|, |l| <= 2^-17 |x|.  (ml and lm
// together reach 2^-24, half a unit of the product: both operands 1 + 2^-8 - 2^-17.)
#pragma once
#include "gemm.hpp"
#include "gemm_tiles.hpp"

namespace gmlp {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Two floats -> two bf16, round to nearest even, packed (low half: the first).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const bf16x2 p = __builtin_convertvector(f32x2{a, b}, bf16x2);
  return __builtin_bit_cast(uint32_t, p);
}
// The three parts of a pair.  The residuals are exact: x - h has at most 17 significant bits, and so on.
constexpr float SPLIT_SCALE = 65536.0f;  // of each operand
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&p)[3]) {
  a *= SPLIT_SCALE;
  b *= SPLIT_SCALE;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    p[i] = pack_bf16(a, b);
    if (i < 2) {
      a -= __builtin_bit_cast(float, p[i] << 16);
      b -= __builtin_bit_cast(float, p[i] & 0xffff0000u);
    }
  }
}

// One operand tile of ROWS rows by BK = 32 reduction elements: float32 in registers on the way in,
// three bf16 planes in LDS.
//   KC plane: row r at byte 64 r, 16-byte chunk c (8 reduction elements) at position c ^ ((r >> 2) & 3)
//   KS plane: reduction row k at byte 2 ROWS k, chunk c (8 rows) at position c ^ swz(k); the 4 (times 2)
//             reduction rows that a transposing read gathers lie in distinct banks
template <int ROWS, bool KS, int NT>
struct SplitTile {
  static constexpr int BK = 32;
  static constexpr int PLANE = ROWS * BK * 2, BYTES = 3 * PLANE;
  static constexpr int CHUNKS = ROWS * BK / 8 / NT;  // 8-element chunks per thread
  static_assert(ROWS * BK / 8 % NT == 0 && CHUNKS >= 1, "chunks divide evenly over the workgroup");
  static constexpr int CPR = KS ? ROWS / 8 : BK / 8;  // chunks per LDS row

  static __device__ __forceinline__ int swz(int row) {
    if (!KS) return (row >> 2) & 3;
    if (ROWS >= 128) return (4 * (row & 3)) ^ (2 * ((row >> 3) & 1));
    return (2 * ((row >> 1) & 1)) ^ (4 * ((row >> 3) & 1));
  }

  const float* ptr[CHUNKS];
  int kofs[CHUNKS];  // reduction index of the chunk within the tile (KC: of its first element)

  // Rows beyond the matrix read the last valid ones: they only feed output that is not stored.
  __device__ __forceinline__ void start(const float* p, int ld, int r0, int k0, int rtot, int tid) {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int q = tid + i * NT, row = q / CPR, c = q % CPR;
      if (KS) {
        kofs[i] = row;
        ptr[i] = p + (size_t)(k0 + row) * ld + min(r0 + c * 8, rtot - 8);
      } else {
        kofs[i] = c * 8;
        ptr[i] = p + (size_t)min(r0 + row, rtot - 1) * ld + (k0 + c * 8);
      }
    }
  }
  // Chunk i of the tile that the pointers stand at into registers, then on to the next tile.  kleft:
  // reduction elements left from the tile's start; what lies beyond them reads as zeros (from `zeros`).
  __device__ __forceinline__ void load1(f32x4 (&raw)[2], int i, int ld, int kleft, const float* zeros) {
    const float* p = kofs[i] < kleft ? ptr[i] : zeros;
    raw[0] = *(const f32x4*)p;
    raw[1] = *(const f32x4*)(p + 4);
    ptr[i] += KS ? (size_t)BK * ld : (size_t)BK;
  }
  // Chunk i, split, into its place in the three planes.
  static __device__ __forceinline__ void store(char* lds, const f32x4 (&raw)[2], int i, int tid) {
    const int q = tid + i * NT, row = q / CPR, c = q % CPR;
    u32x4 o[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t p[3];
      split_pair(raw[j / 2][2 * (j % 2)], raw[j / 2][2 * (j % 2) + 1], p);
#pragma unroll
      for (int s = 0; s < 3; ++s) o[s][j] = p[s];
    }
    char* at = lds + row * (CPR * 16) + ((c ^ swz(row)) << 4);
#pragma unroll
    for (int s = 0; s < 3; ++s) *(u32x4*)(at + s * PLANE) = o[s];
  }
  // Fragment of plane s for v_mfma_f32_16x16x32_bf16: lane l carries row row0 + l % 16 and reduction
  // elements 8 (l / 16) .. + 7.
  static __device__ __forceinline__ bf16x8 frag(const char* lds, int s, int row0, int lane) {
    const char* t = lds + s * PLANE;
    if constexpr (!KS) {
      const int row = row0 + (lane & 15);
      return *(const bf16x8*)(t + row * 64 + (((lane >> 4) ^ swz(row)) << 4));
    } else {
      const int r = lane & 15, k = 8 * (lane >> 4) + (r >> 2), n = row0 + 4 * (r & 3);
      const char* a0 = t + k * (ROWS * 2) + (((n >> 3) ^ swz(k)) << 4) + ((n & 7) << 1);
      // reduction row k + 4: ROWS >= 128 the same position; 64 rows: bit 1 of (k >> 1) does not change with 4
      i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)a0);
      i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(a0 + 4 * (ROWS * 2)));
      i16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(bf16x8, both);
    }
  }
};

}  // namespace gmlp
