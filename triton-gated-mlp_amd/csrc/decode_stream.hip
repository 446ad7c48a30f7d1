// Skinny-M (M <= 32) weight-streaming kernels, HBM-bound: every weight byte is fetched once, in
// row segments of 128, 256 or 512 bytes moved global -> LDS without passing through registers.
//
// One persistent workgroup of three or four wavefronts per CU.  The workgroup takes blocks of weight rows
// that share one set of token operands: 16 to 80 rows of W_gate and as many of W_up (GATED), or 8, 16,
// 32 or 64 consecutive rows of W_down.  Whole blocks go round-robin over the workgroups, the rows that
// do not fill a last round are shared out evenly as one partly empty block each.  Its wavefronts split
// the reduction range in near-equal runs of chunks (64 to 256 elements) and combine their partial
// sums through LDS at the end of each block (fixed order, so the result is deterministic).  Each
// wavefront runs a private ring of 2 to 8 LDS slots; a slot holds one stage = one chunk of the
// block's weight rows.  The matching token-row operands (x or H, L2-resident)
// are fetched straight into registers, as many stages ahead: one 16-token tile for M <= 16, two
// beyond (MT; the weight fragment read from LDS then feeds two MFMAs).  The stream of stages runs on
// across block boundaries, so the ring never drains; the loads of stages past the end go nowhere (an offset beyond the
// descriptor reads as zero and moves no data), which keeps the in-flight count constant.  (Fetching the last stage
// again instead: whole forward M=24, K=4096, N=11008 55.8 us for 53.4, M=16, K=8192, N=28672 214.0 for 211.6.)
//
// Which block (chosen in launch_decode_stream; kernel times, us, fp16): the height decides what a block
// costs in token operands and how well it fits a CU's share of the rows; the row segment of a stage (SEGB)
// how evenly the chunks divide over the wavefronts (16 chunks of 256 elements at K = 4096: 6, 5 and 5; 64 of
// 64: 22, 21 and 21), how soon the first MFMA can start, and how finely the ring's slots take up what the
// loads in flight leave.  512- -> 128-byte segments, W_gate / W_up, 16 rows a block: K=2048, N=8192 M=8
// 17.4 -> 14.6, M=16 19.1 -> 15.4; K=1024, N=4096 9.3 -> 7.1, 10.1 -> 7.6.  Bytes in flight do not decide once full
// slots hold 96 KiB per CU: four, six and eight wavefronts with 128 to 144 KiB were no faster on any of eleven
// widths.  Where a CU's share leaves slots partly empty they do: four wavefronts then, see launch_decode_stream.
//
//   GATED:   H[m, r] = act(x.W_gate[r] + b_gate[r]) * (x.W_up[r] + b_up[r])      (r over N)
//   !GATED:  Y[m, r] = H.W_down[r] + b_down[r]                                   (r over K)
//
// LDS layout of a slot: regions of 16 (or 8, RR) rows x SEGB bytes; the 16-byte chunk c of row r is stored at
// position c ^ r (128-byte segments, two rows to all banks: c ^ (r / 2)), so the 16 lanes that read one
// chunk index of 16 different rows for v_mfma_f32_16x16x32 hit 16 different bank groups.
//
// All vector-memory loads of the main loop are written as assembly and ordered by explicit
// s_waitcnt vmcnt(N): the compiler does not see them, so it cannot serialise them either (the
// build checks the generated assembly for uses of a load's destination ahead of its wait).
#include "launch.hpp"
#include "lds_dma.hpp"

namespace gmlp {

typedef float f32x4v __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma16x;
template <>
struct Mfma16x<f16> {
  static __device__ __forceinline__ f32x4v run(f16x8 a, f16x8 b, f32x4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16x<bf16> {
  static __device__ __forceinline__ f32x4v run(bf16x8 a, bf16x8 b, f32x4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

constexpr int DS_MAX_LDS = 160 * 1024;
constexpr int DS_MIN_RED = 768;               // a chunk for every wavefront (three of 256 elements, four of 64)
constexpr uint32_t DS_NOWHERE = 0x80000000u;  // voffset beyond any operand (operands are < 2 GiB)
constexpr int DS_WIDE_SEGMENT_MAX_M = 20;     // see ds_tall_gated, ds_short_segments
constexpr int DS_H_TILED_MIN_M = 10;           // H goes out in fragment order above this many token rows

struct StreamArgs {
  const void* x;      // [M, ldx] token rows (x or H)
  const void* w[2];   // [R, red] weight matrices
  const void* bias[2];
  void* out;          // [M, ldo]
  int M, R, red, ldx, ldo;
  int act;            // Act code (GATED only)
  int tiled;          // H (GATED: out, otherwise: x) is in fragment order, see ds_h_tiled()
};

typedef int i32x4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane into registers; completion is tracked by the caller (wait_vmem_keep).
__device__ __forceinline__ i32x4 load16_async(buffer_rsrc r, uint32_t voffset, uint32_t soffset) {
  i32x4 v;
  asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen"
               : "=v"(v)
               : "v"(voffset), "s"(r), "s"(soffset)
               : "memory");
  return v;
}
// s_waitcnt vmcnt(N) that also "defines" the registers a stage's token operands arrive in, so no use
// of them can be scheduled above the wait.  The other statements issue no instruction: volatile asm
// statements keep their order, so they tie the other registers to the same point.
template <int N, int NX>
__device__ __forceinline__ void wait_vmem_keep(i32x4 (&x)[NX]) {
  static_assert(NX % 2 == 0, "pairs");
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(x[0]), "+v"(x[1]) : "n"(N) : "memory");
#pragma unroll
  for (int i = 2; i < NX; i += 2) asm volatile("" : "+v"(x[i]), "+v"(x[i + 1]) : : "memory");
}

// A workgroup barrier that orders LDS accesses only: loads in flight stay in flight.
__device__ __forceinline__ void ds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// HALVES: regions per matrix and stage.
// MT:   tiles of 16 token slots (M <= 16 * MT).
// SEGB: bytes of a weight row per stage, 512, 256 or 128.
// DS_RD: ring slots per wavefront and stages in flight.
// TAIL: the reduction length need not be a multiple of the chunk (only of 8): the 16-byte pieces of the
//       last chunk that lie beyond the row's end are pushed out of the descriptors, weights and token
//       operands, and read as zeros.  An instance of its own: the others have no such selects.
// RR:   rows of a region: 16, or 8, which the MFMA's rows 8 to 15 read again, for shares of the rows (see share)
//       of no more than 8: of a 16-row slot only half would hold weights.
// NW:   wavefronts.
// (wg and G, the workgroup's number and count, are members and not read where they are used: the compiler then spills
// twice the scalars, and over 1247 shapes the forward takes 1.02 of the time, small ones up to 1.15.  The same body as one
// function takes 1.00 of it, 1.01 to 1.02 with two token tiles.)
template <typename T, bool GATED, int HALVES, int MT, int SEGB, int DS_RD, bool TAIL, int RR, int NW>
struct StreamBody {
  typedef typename Traits<T>::vec8 vec8;
  static_assert(SEGB == 512 || SEGB == 256 || SEGB == 128, "row segment of a stage");
  static constexpr int NREG = (GATED ? 2 : 1) * HALVES;  // regions per stage
  static constexpr int REGION = RR * SEGB;               // bytes of a region
  static constexpr int CH = SEGB / 2;                    // reduction elements per stage
  static constexpr int KS = CH / 32;                     // MFMA steps per stage
  static constexpr int CPR = SEGB / 16;                  // 16-byte chunks per row segment
  static constexpr int LPR = REGION / 1024;  // load instructions per region (64 lanes x 16 bytes each)
  // The token operands in flight live in VGPRs that the loads fill asynchronously.  Were there not
  // enough of the 256 left beside them, the compiler would park them elsewhere right after the
  // load instruction, before the data has arrived.
  static_assert(DS_RD * KS * MT * 4 <= 192, "token operands in flight must leave room in the VGPRs");
  // weight rows (per matrix) a block advances by
  static constexpr int BLOCK_ROWS = RR * HALVES;
  static constexpr int SLOT = NREG * REGION;
  static constexpr int LPS = KS * MT + NREG * LPR;  // load instructions per stage (token operands + weights)
  // A stage is complete when no more than the DS_RD - 1 younger stages are in flight.  vmcnt has 6
  // bits: where that count exceeds 63 the wait also covers the first token-operand loads of the
  // next stage (issued right behind the awaited weights, and loads return in order).
  static constexpr int YOUNGER = (DS_RD - 1) * LPS < 63 ? (DS_RD - 1) * LPS : 63;
  static_assert((DS_RD - 1) * LPS - YOUNGER <= KS * MT, "the wait may only reach into the next stage's token operands");
  // Partial sums change hands through LDS in two alternating buffers, or, where LDS does not hold
  // two, in one buffer with a second barrier behind its readers.
  static constexpr int RING_BYTES = NW * DS_RD * SLOT;
  static constexpr int PART_FLOATS = (NW - 1) * NREG * MT * 256;
  static constexpr int PARITIES = RING_BYTES + 2 * PART_FLOATS * 4 <= DS_MAX_LDS ? 2 : 1;
  static constexpr int LDS_BYTES = RING_BYTES + PARITIES * PART_FLOATS * 4;
  static_assert(LDS_BYTES <= DS_MAX_LDS, "a workgroup has 160 KiB of LDS");

  static __device__ __forceinline__ int swz(int r) { return SEGB == 128 ? r >> 1 : r; }

  int lane, wave, wg, G;
  uint32_t lds_base;
  char* ring;
  float* part;  // [parities][waves-1][NREG][MT][64][4]
  int full, t_begin, t_end, my_blocks, c0, spb, total, rot;
  int r16, kg;
  uint32_t woff[LPR], xoff[MT];
  int wrow[LPR];    // row of the region that load q of this lane fetches
  int wchunk[LPR];  // TAIL: and its 16-byte piece of the row's segment
  bool tiled_x;
  uint32_t xq, pitch;
  i32x4 xf[DS_RD][KS * MT];  // [stage in flight][MFMA step q][token tile]
  f32x4v acc[NREG][MT];

  // Blocks of BLOCK_ROWS weight rows go round-robin over the workgroups (block b, b + G, ...: at any
  // time the chip streams one contiguous band of rows) for as many rounds as every workgroup gets a
  // whole block.  The rows left over (the tail) are shared out evenly instead, in multiples of 4
  // (what one lane stores), so that every CU streams the same number of bytes whatever R is: a
  // workgroup's tail share [t_begin, t_end) is one last block with fewer valid rows, the loads of
  // the others go nowhere and their results are not stored.
  __device__ __forceinline__ void share(const StreamArgs& a, int wg_, int G_) {
    wg = wg_;
    G = G_;
    full = a.R / BLOCK_ROWS / G;
    const int tail0 = full * G * BLOCK_ROWS, tail_rows = a.R - tail0;
    t_begin = tail0 + ((wg * tail_rows / G) & ~3);
    t_end = wg + 1 == G ? a.R : tail0 + (((wg + 1) * tail_rows / G) & ~3);
    my_blocks = full + (t_end - t_begin + BLOCK_ROWS - 1) / BLOCK_ROWS;
  }
  // first row and number of existing rows (BLOCK_ROWS or more: all) of this workgroup's j-th block
  __device__ __forceinline__ void block_rows(int j, int& row0, int& valid) const {
    if (j < full) {
      row0 = (wg + j * G) * BLOCK_ROWS;
      valid = BLOCK_ROWS;
    } else {
      row0 = t_begin + (j - full) * BLOCK_ROWS;
      valid = t_end - row0;
    }
  }

  // A wavefront's part in the share of workgroup wg_ of G_.
  __device__ __forceinline__ void start(const StreamArgs& a, char* smem, int wave_, int wg_, int G_) {
    lane = threadIdx.x & 63;
    wave = wave_;
    lds_base = (uint32_t)(uintptr_t)(lds_void*)smem + wave * (DS_RD * SLOT);
    ring = smem + wave * (DS_RD * SLOT);
    part = (float*)(smem + RING_BYTES);
    share(a, wg_, G_);
    const int chunks = TAIL ? (a.red + CH - 1) / CH : a.red / CH;
    // wavefront w reduces chunks [c0, c0 + spb)
    c0 = (chunks * wave) / NW;
    spb = (chunks * (wave + 1)) / NW - c0;
    total = my_blocks * spb;
    // Workgroup b starts each block at chunk b % spb of its wavefronts' ranges and wraps around (a
    // sum does not mind the order).  Without it every workgroup on the chip reads the same offset
    // along its rows at the same time, and for a power-of-two row pitch (W_gate, W_up of the usual
    // hidden sizes) those addresses crowd onto a few memory channels: 154 -> 142 us at K = 8192.
    rot = wg % spb;

    // Per-lane byte offsets: weights, LPR load instructions per region (1024 / SEGB rows each);
    // token operands, the 16 bytes of token row 16 t + lane%16 this lane feeds to the MFMAs of tile t.
    r16 = lane & 15;
    kg = lane >> 4;
#pragma unroll
    for (int q = 0; q < LPR; ++q) {
      int row = (64 / CPR) * q + lane / CPR, pos = lane % CPR;
      wrow[q] = row;
      wchunk[q] = pos ^ swz(row);
      woff[q] = (uint32_t)(row * a.red + (pos ^ swz(row)) * 8) * 2u;
    }
    tiled_x = !GATED && a.tiled;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if (tiled_x) {
        // [red/8][16 MT token slots][8 elements]: the 8-element group kg of a fragment is 256 MT
        // bytes after the previous one (for MT = 1 a fragment is one contiguous KiB)
        xoff[t] = (uint32_t)(kg * (256 * MT) + t * 256 + r16 * 16);
      } else {
        int xr = 16 * t + r16 < a.M ? 16 * t + r16 : a.M - 1;  // rows past M repeat the last token row
        xoff[t] = (uint32_t)(xr * a.ldx + kg * 8) * 2u;
      }
    }
    xq = tiled_x ? 1024u * MT : 64u;  // from one MFMA's token operand to the next
    pitch = (uint32_t)a.red * 2u;
#pragma unroll
    for (int g = 0; g < NREG; ++g)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[g][t] = f32x4v{0.f, 0.f, 0.f, 0.f};
  }

  // Exact sizes: an offset past the end reads as zero instead of touching memory.  (Put together from the kernel's
  // arguments where they are used: carried along as members they came to lie in VGPRs.)
  __device__ __forceinline__ buffer_rsrc token_rsrc(const StreamArgs& a) const {
    return make_rsrc(a.x, !GATED && a.tiled ? (uint32_t)(16 * MT) * (uint32_t)a.red * 2u : (uint32_t)a.M * (uint32_t)a.ldx * 2u);
  }
  // of region g of a stage: GATED: matrix g / HALVES, rows RR (g % HALVES) on of the block; otherwise rows
  // RR g on of the block of W_down
  __device__ __forceinline__ buffer_rsrc weight_rsrc(const StreamArgs& a, int g) const {
    return make_rsrc(a.w[GATED ? g / HALVES : 0], (uint32_t)a.R * (uint32_t)a.red * 2u);
  }

  // Stage i of this wavefront's stream: where in the block and along the reduction it is, and how many
  // 16-byte pieces of its segment lie inside the row (0: no such stage).
  __device__ __forceinline__ void stage(const StreamArgs& a, int i, int& row0, int& valid, uint32_t& koff, int& pieces) const {
    const bool past = i >= total;
    const int ii = past ? total - 1 : i;
    const int j = ii / spb;
    int c = ii - j * spb + rot;
    c = c < spb ? c : c - spb;
    block_rows(j, row0, valid);
    koff = (uint32_t)((c0 + c) * CH) * 2u;
    pieces = past ? 0 : TAIL ? (a.red - (c0 + c) * CH) / 8 : CPR;
    valid = past ? 0 : valid;
  }
  // Its token operands into xf[u].
  __device__ __forceinline__ void issue_tokens(const StreamArgs& a, int i, int u) {
    int row0, valid, pieces;
    uint32_t koff;
    stage(a, i, row0, valid, koff, pieces);
    // token operand of the stage's q-th MFMA step: 64 bytes further along each row of x, or the
    // next fragment of H (a stage of CH elements x 16 MT token slots)
    const uint32_t xstage = tiled_x ? koff * (16u * MT) : koff;
#pragma unroll
    for (int q = 0; q < KS; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xf[u][q * MT + t] = load16_async(token_rsrc(a), (TAIL ? q * 4 + kg < pieces : pieces > 0) ? xoff[t] : DS_NOWHERE, xstage + q * xq);
  }
  // Its weights into ring slot u.
  __device__ __forceinline__ void issue_weights(const StreamArgs& a, int i, int u) {
    int row0, valid, pieces;
    uint32_t koff;
    stage(a, i, row0, valid, koff, pieces);
    uint32_t slot = lds_base + (uint32_t)u * SLOT;
    uint32_t woffs = (uint32_t)row0 * pitch + koff;
#pragma unroll
    for (int g = 0; g < NREG; ++g) {
      const int first = GATED ? RR * (g % HALVES) : RR * g;  // region's first row within the block
      const int valid_g = valid - first;
#pragma unroll
      for (int q = 0; q < LPR; ++q)
        load16_to_lds<true>(weight_rsrc(a, g),
                            wrow[q] < valid_g && (!TAIL || wchunk[q] < pieces) ? woff[q] : DS_NOWHERE,
                            woffs + (uint32_t)first * pitch, slot + g * REGION + q * 1024);
    }
  }
  __device__ __forceinline__ void issue_stage(const StreamArgs& a, int i, int u) {
    issue_tokens(a, i, u);
    issue_weights(a, i, u);
  }

  // Block blk's sums, this wavefront's (0) and those that the others left in LDS, and what comes of them.  A
  // lane holds, per token tile t, token row 16 t + lane%16 and, per region, weight rows 4*(lane/16) + r of
  // the region.
  __device__ __forceinline__ void finish_block(const StreamArgs& a, int blk, const float* pp) {
    int row0, valid;
    block_rows(blk, row0, valid);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int tok = 16 * t + r16;
      if (!((GATED && a.tiled) || tok < a.M)) continue;
      float v[NREG][4];
#pragma unroll
      for (int g = 0; g < NREG; ++g) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[g][r] = acc[g][t][r];
#pragma unroll
        for (int w = 0; w < NW - 1; ++w) {
          f32x4v o = *(const f32x4v*)(pp + ((w * NREG + g) * MT + t) * 256 + lane * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[g][r] += o[r];
        }
        // this lane's four rows of the region, as rows of the block
        const int first = (GATED ? RR * (g % HALVES) : RR * g) + 4 * kg;
        const T* bias = (const T*)a.bias[GATED ? g / HALVES : 0];
        if (bias && 4 * kg < RR && first < valid) add_w<T, 4>(bias + row0 + first, v[g]);
      }
      if (GATED) {
#pragma unroll
        for (int hf = 0; hf < HALVES; ++hf) {
          const int first = RR * hf + 4 * kg;
          const int r0 = row0 + first;
          float res[4];
          act_fwd_w<4>(a.act, v[hf], res);
#pragma unroll
          for (int r = 0; r < 4; ++r) res[r] *= v[HALVES + hf][r];
          // Fragment order: H goes out the way the down projection's MFMAs take it in,
          // [N/8][16 MT token slots][8 elements], so that a token-operand fragment there is
          // 4 runs of 256 MT bytes (one contiguous KiB for MT = 1) instead of 16 row pieces
          // of 64 bytes.  All slots are written (slots past M repeat the last token), so
          // nothing uninitialised is multiplied.
          if (4 * kg < RR && first < valid)
            store_w<T, 4>(a.tiled ? (T*)a.out + ((size_t)(r0 >> 3) * (16 * MT) + tok) * 8 + (r0 & 7)
                                  : (T*)a.out + (size_t)tok * a.ldo + r0,
                          res);
        }
      } else {
#pragma unroll
        for (int g = 0; g < NREG; ++g)
          if (4 * kg < RR && RR * g + 4 * kg < valid)
            store_w<T, 4>((T*)a.out + (size_t)tok * a.ldo + row0 + RR * g + 4 * kg, v[g]);
      }
    }
  }

  // All stages, the first DS_RD of which are in flight.  Loads of stages past the end may be in flight behind it.
  __device__ __forceinline__ void run(const StreamArgs& a) {
    int in_block = 0, blk = 0;
    for (int i0 = 0; i0 < total; i0 += DS_RD) {
#pragma unroll
      for (int u = 0; u < DS_RD; ++u) {
        const int i = i0 + u;
        if (i < total) {
          wait_vmem_keep<YOUNGER, KS * MT>(xf[u]);
          const char* slot = ring + u * SLOT;
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            int pos = ((ks * 4 + kg) ^ swz(RR == 16 ? r16 : r16 & (RR - 1))) << 4;
#pragma unroll
            for (int g = 0; g < NREG; ++g) {
              vec8 wf = *(const vec8*)(slot + g * REGION + (RR == 16 ? r16 : r16 & (RR - 1)) * SEGB + pos);
#pragma unroll
              for (int t = 0; t < MT; ++t)
                acc[g][t] = Mfma16x<T>::run(wf, __builtin_bit_cast(vec8, xf[u][ks * MT + t]), acc[g][t]);
            }
          }
          // The MFMAs above consumed every LDS read of this slot, so it can be refilled.
          issue_stage(a, i + DS_RD, u);

          if (++in_block == spb) {
            // Block finished: wavefronts 1.. hand their partial sums to wavefront 0.
            in_block = 0;
            float* pp = part + (PARITIES == 2 ? (blk & 1) * PART_FLOATS : 0);
            if (wave > 0) {
#pragma unroll
              for (int g = 0; g < NREG; ++g)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                  *(f32x4v*)(pp + (((wave - 1) * NREG + g) * MT + t) * 256 + lane * 4) = acc[g][t];
            }
            ds_barrier();
            if (wave == 0) finish_block(a, blk, pp);
            // one buffer: nobody writes the next block's partial sums before wavefront 0 has read these
            if (PARITIES == 1) ds_barrier();
#pragma unroll
            for (int g = 0; g < NREG; ++g)
#pragma unroll
              for (int t = 0; t < MT; ++t) acc[g][t] = f32x4v{0.f, 0.f, 0.f, 0.f};
            ++blk;
          }
        }
      }
    }
  }
};

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
  // one workgroup per CU, each with its share of the rows (a partly empty block when that is less
  // than a block); fewer workgroups when a share would be under 8 rows
  int grid = a.R / 8 < num_cu ? a.R / 8 : num_cu;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), LDS, s, a);
  return hipGetLastError();
}
template <typename T, bool GATED, int HALVES, int MT, int SEGB, int RD, int RR = 16, int NW = 3>
static hipError_t launch_stream(const StreamArgs& a, int num_cu, hipStream_t s) {
  if constexpr (SEGB > 128)  // (rows of whole 128-byte lines are a multiple of 64 elements)
    if (a.red % (SEGB / 2) != 0) return launch_stream_tail<T, GATED, HALVES, MT, SEGB, RD, true, RR, NW>(a, num_cu, s);
  return launch_stream_tail<T, GATED, HALVES, MT, SEGB, RD, false, RR, NW>(a, num_cu, s);
}

// Layout of the intermediate H between the two kernels.  Row-major [M, N] costs the down projection
// M pieces of 64 bytes per token-operand fragment, fragment order always one KiB (16 token slots):
// cheaper from about half-full upwards.  Two token tiles always use fragment order.
static int ds_h_tiled(int M) { return M > DS_H_TILED_MIN_M ? 1 : 0; }

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
