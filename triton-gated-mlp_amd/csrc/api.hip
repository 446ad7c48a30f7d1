// extern "C" entry points of libgmlp.so (declared in include/gmlp.h): argument validation,
// tile-class selection and kernel launches.  All validation happens before the first HIP call,
// so the error paths can be exercised on a machine without a GPU.
#include "gmlp.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <vector>

#include "launch.hpp"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

#define GMLP_REQUIRE_PTR(p)                                                         \
  if ((p) == nullptr) return fail(GMLP_EINVAL, "%s: argument '%s' is NULL", __func__, #p)
#define GMLP_REQUIRE_ALIGNED(p)                                                     \
  if ((p) != nullptr && !aligned16(p))                                              \
  return fail(GMLP_EALIGN, "%s: argument '%s' is not 16-byte aligned", __func__, #p)
#define GMLP_REQUIRE_DTYPE(d)                                                       \
  if ((d) != GMLP_F16 && (d) != GMLP_BF16 && (d) != GMLP_F32)                       \
  return fail(GMLP_EINVAL, "%s: dtype %d is not GMLP_F16/GMLP_BF16/GMLP_F32", __func__, (int)(d))

#define GMLP_REQUIRE_ACT(a)                                                         \
  if ((a) < 0 || (a) >= gmlp::ACT_COUNT)                                            \
  return fail(GMLP_EINVAL, "%s: act %d is not one of the GMLP_ACT_* codes", __func__, (int)(a))

static_assert(GMLP_COLSUM_STATIC_MAX_C == gmlp::COLSUM_STATIC_MAX_C, "public limit of gmlp_colsum_static");
static_assert((int)GMLP_ACT_SILU == (int)gmlp::ACT_SILU && (int)GMLP_ACT_GELU == (int)gmlp::ACT_GELU &&
                  (int)GMLP_ACT_RELU == (int)gmlp::ACT_RELU && (int)GMLP_ACT_LEAKY_RELU == (int)gmlp::ACT_LEAKY_RELU &&
                  (int)GMLP_ACT_SIGMOID == (int)gmlp::ACT_SIGMOID && (int)GMLP_ACT_TANH == (int)gmlp::ACT_TANH &&
                  (int)GMLP_ACT_IDENTITY == (int)gmlp::ACT_IDENTITY && gmlp::ACT_COUNT == 7,
              "device activation codes are the public ones");

const int64_t kMaxDim = (int64_t)1 << 30;

int check_dims(const char* fn, int64_t M, int64_t K, int64_t N) {
  if (M < 1 || K < 1 || N < 1) return fail(GMLP_ESHAPE, "%s: M, K, N must be >= 1 (got %lld, %lld, %lld)", fn,
                                           (long long)M, (long long)K, (long long)N);
  if (M > kMaxDim || K > kMaxDim || N > kMaxDim || M * N >= ((int64_t)1 << 40) ||
      M * K >= ((int64_t)1 << 40))
    return fail(GMLP_ESHAPE, "%s: dimension too large", fn);
  return 0;
}

int check_mult8(const char* fn, const char* name, int64_t v) {
  if (v % 8 != 0)
    return fail(GMLP_ESHAPE, "%s: %s = %lld must be a multiple of 8 (16-byte rows)", fn, name, (long long)v);
  return 0;
}

int make_dropout(const char* fn, float p, uint64_t seed, uint64_t offset, gmlp::DropoutParams* d) {
  if (!(p >= 0.0f) || !(p < 1.0f))
    return fail(GMLP_EINVAL, "%s: dropout_p = %g must satisfy 0 <= p < 1", fn, (double)p);
  d->enabled = p > 0.0f ? 1 : 0;
  double t = std::floor((double)p * 4294967296.0);
  d->threshold = t >= 4294967295.0 ? 4294967295u : (uint32_t)t;
  d->scale = 1.0f / (1.0f - p);
  d->seed_lo = (uint32_t)seed;
  d->seed_hi = (uint32_t)(seed >> 32);
  d->off_lo = (uint32_t)offset;
  d->off_hi = (uint32_t)(offset >> 32);
  return 0;
}

// Calls f(T{}) with T = the storage type named by `dtype` (already validated).
template <typename F>
hipError_t by_dtype(int dtype, F&& f) {
  if (dtype == GMLP_F16) return f(gmlp::f16{});
  if (dtype == GMLP_BF16) return f(gmlp::bf16{});
  return f(float{});
}

int hip_result(const char* fn, hipError_t e) {
  if (e == hipSuccess) return GMLP_OK;
  return fail(GMLP_EHIP, "%s: HIP error %d (%s)", fn, (int)e, hipGetErrorString(e));
}

// Scheduling groups of 8 tile-rows when the A operand (rows x red) is the smaller one, of 8
// tile-columns (negative) when B (cols x red, `sets` of them) is: see tile_of_grouped.
int pick_group(int64_t rows, int64_t cols, int sets = 1) { return sets * cols < rows ? -8 : 8; }

// Compute units of the current device.
int num_cu() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Accelerator dies (XCDs, each with an L2 of its own) behind the current device: the hardware
// deals consecutive workgroup ids round-robin to them.  A gfx950 XCD has 32 active compute units,
// so a whole MI355X shows 8 and a partition of it 4, 2 or 1.
int num_xcd() {
  int n = num_cu() / 32;
  return n < 1 ? 1 : n > 8 ? 8 : n;
}

// The GEMMs of a gated MLP (operand layouts, epilogues: launch.hpp).
enum GemmKind { GATEUP, LINEAR, DH, DX, DW };

const int64_t kMaxSplits = 16;

// How a GEMM runs: tile class, and number of workgroups that share an output tile, each reducing a
// contiguous range of reduction tiles (1: no split).
struct GemmPlan {
  int tile_class;
  int splits;
  double us;  // estimate
};

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// float32: tile class and number of workgroups per tile (splits), by estimated time: rounds of 2
// (128x128 tiles) or 3 (64x64; 2 with two accumulator sets) workgroups per CU, each reduction tile at what
// it takes with that many workgroups on a CU, a last round as long as the CUs with the most, a little
// less where they are few.  A split reduction pays a second launch and the partial sums' round trip
// through the caches.  One least-squares fit to the launches of five GEMMs of 70 shapes (M 32 to 6000,
// widths 40 to 14400, both classes, 1 to 16 splits): standard deviation of the estimates 6 %, what it picks
// costs 0.4 % over the fastest on average.  What that is worth at M=2048, K=1024, N=2816: down projection
// on 128x128 tiles (128 of them) unsplit 161 us, in 4 splits 94, 64x64 unsplit 105; dX 302 / 162 / 199.
// us per reduction tile with 1, 2, 3 workgroups on a CU; us of an epilogue
const double kF32R128[] = {1.802, 2.885}, kF32R64[] = {0.721, 1.167, 1.549}, kF32R64x2[] = {1.271, 1.930};
const double kF32E128 = 2.597, kF32E64 = 0.925;
const double kF32Launch = 4.05, kF32Traffic = 0.345e-6;  // us of a launch; of a byte of partial sums
GemmPlan plan_f32(int64_t tiles128, int64_t tiles64, int64_t red_tiles, int sets, double out_bytes, int64_t max_splits,
                  double split_us) {
  GemmPlan best = {gmlp::TILE_F32_128, 1, 1e30};
  const int64_t cus = num_cu();
  auto consider = [&](int tile_class, int64_t tiles, int64_t splits) {
    const bool big = tile_class == gmlp::TILE_F32_128;
    const double* r = big ? kF32R128 : sets == 2 ? kF32R64x2 : kF32R64;
    const int64_t cap = big || sets == 2 ? 2 : 3, wgs = tiles * splits, k = cdiv(red_tiles, splits), rest = wgs % (cus * cap);
    const double e = big ? kF32E128 : kF32E64;
    double us = kF32Launch + (double)(wgs / (cus * cap)) * ((double)k * r[cap - 1] + e);
    if (rest > 0) {
      const int64_t per = cdiv(rest, cus);
      const double f = (double)rest / (double)cus - (double)(per - 1);
      us += (double)k * (r[per - 1] - 0.114 * (1.0 - f) * (r[per - 1] - (per > 1 ? r[per - 2] : 0.0))) + e;
    }
    if (splits > 1) us += split_us + kF32Traffic * (double)splits * out_bytes * sets;
    if (us < best.us) best = GemmPlan{tile_class, (int)splits, us};
  };
  for (int64_t s = 1; s <= std::max<int64_t>(1, std::min(max_splits, red_tiles / 4)); ++s) {
    if (s > 1 && cdiv(red_tiles, cdiv(red_tiles, s)) != s) continue;  // rounding up would leave splits empty
    consider(gmlp::TILE_F32_128, tiles128, s);
    consider(gmlp::TILE_F32_64, tiles64, s);
  }
  return best;
}
// What a split costs beside its traffic: 1.7 us on the GPU, and the rest is what the second launch costs the
// host, which bounds passes this small.  A forward down projection pays that twice: nothing else in its
// pass is split at such sizes (training step at M=K=N=512 89.4 us with one launch, 92.4 with two).
const double kSplitF32 = 4.9, kSplitF32Linear = 8.9;
GemmPlan plan_f32(int64_t rows, int64_t cols, int64_t red_tiles, int kind, int64_t max_splits) {
  const int sets = kind == GATEUP ? 2 : 1;
  return plan_f32(cdiv(rows, 128) * cdiv(cols, 128 / sets), cdiv(rows, 64) * cdiv(cols, 64), red_tiles, sets,
                  (double)rows * (double)cols * 4.0, max_splits, kind == LINEAR ? kSplitF32Linear : kSplitF32);
}

// Stream-K plan for a grid of `tiles` large output tiles with `kt` 64-wide reduction tiles each
// (tiles of all problems of a grouped launch together).  The tiles beyond the last whole round of
// workgroups (one per compute unit) are shared out by reduction range when that beats running them
// as a thinly filled round: a round filled to the fraction f costs about 0.6 + 0.4 f of a full one
// (kLarge has the later fit, 0.69 + 0.31 f) against f with stream-K, plus the partial sums' round trip
// through memory and the second launch (about 45 us, i.e. 30 reduction tiles' time): worth it when
// (1 - f) * kt > 50.
// Every stream-K workgroup gets at least 8 reduction tiles.
// A grid of less than one round that fills more than half of the chip is left alone unless its tiles
// divide into whole pieces (`first_round`: false for the weight gradients, which keep the plan): even
// ranges straddle tiles there, two partial stores per workgroup, and the busy CUs of the plain launch
// clock higher.  Down projections of 160 tiles: 322 to 330 us shared out, 264 to 275 plain; 192
// tiles: 313 / 292; dX of 192 tiles 362 / 327; 224 tiles 247 / 246.  (96 tiles: 324 / 495.)
struct StreamK {
  int tiles = 0, wgs = 0, chunks = 0;
  size_t ws_bytes = 0;
};
StreamK plan_streamk(int dtype, int64_t tiles, int64_t kt, bool first_round = true) {
  StreamK p;
  const int64_t cus = num_cu(), tail = tiles % cus;
  if (dtype == GMLP_F32 || tail == 0 || kt < 8) return p;
  if ((double)(cus - tail) / (double)cus * (double)kt <= 50.0) return p;
  int64_t wgs = tail * kt / 8;
  if (wgs > cus) wgs = cus;
  if (wgs < 1 || tail * kt >= ((int64_t)1 << 30)) return p;
  p.tiles = (int)tail;
  p.wgs = (int)wgs;
  // A whole number of pieces per tile when that still fills (nearly) all compute units: the
  // workgroups of an XCD then walk neighbouring tiles over the same reduction range and share
  // operand panels in L2 (measured on 128 tiles in halves: the pieces' launch 123 -> 116 us).
  const int64_t per_tile = wgs / tail;
  if (per_tile >= 2 && per_tile * tail * 10 >= wgs * 9 && kt / per_tile >= 8) {
    p.chunks = (int)per_tile;
    p.wgs = (int)(per_tile * tail);
  }
  if (first_round && tiles < cus && 2 * tiles > cus && p.chunks == 0) return StreamK{};
  p.ws_bytes = (size_t)(p.tiles + p.wgs) * 65536 * sizeof(float);  // 256 x 256 accumulators per slot
  return p;
}
// Applies the plan to a launch's arguments when the caller's workspace can hold it.
bool use_streamk(const StreamK& p, gmlp::GemmArgs& ga, void* workspace, size_t workspace_bytes) {
  if (p.tiles == 0 || workspace == nullptr || workspace_bytes < p.ws_bytes) return false;
  ga.sk_tiles = p.tiles;
  ga.sk_wgs = p.wgs;
  ga.sk_chunks = p.chunks;
  ga.sk_ws = (float*)workspace;
  return true;
}

// Output columns (per accumulator set) of a LARGE or WIDE tile; MEDIUM_FULL tiles have half.
int tile_cols(int kind) { return kind == GATEUP ? 128 : 256; }
int64_t red_tiles_of(int kind, int64_t red) { return (kind == DX ? 2 : 1) * cdiv(red, 64); }

// 16-bit types: estimated time of a launch on a tile class, in rounds of workgroups (one per CU, two
// for MEDIUM_FULL).  A round takes kt * r + e us: reduction tiles times the class's rate, and an
// epilogue whose cost is its stores (and, dH, its loads).  A last round filled to the fraction f
// costs base + (1 - base) f of a full one (busy CUs clock higher, but not in proportion; the small
// tiles gain less once a CU has two: base + half up to f = 1/2, 1 at f = 1).  A split reduction adds a
// second launch and the partial sums' round trip.  All constants are one least-squares fit to 3100
// launches (five GEMMs of 89 random shapes, M 33 to 6000, widths 128 to 15000, every class and split;
// standard deviation of the estimates 3 to 12 %); the class chosen cost 1.5 % over the fastest on
// average.  The kernels are faster since (accumulators in place; eight wavefronts on WIDE): of 1929 launches of those, the
// class chosen costs 2.2 % over the fastest for gate/up, 5.9 % for dH and 2.5 % for the down projection.  Constants
// fitted to them cost 1.6, 4.8 and 3.0 %, and no whole pass of 22 moved by more than 1 %: these stay.  What they misjudge, for
// one: gate/up at M=1024, K=2048, N=5632, 55 us estimated on LARGE and 63 on WIDE, takes 52 and 50.
struct TileCost {
  int tile_class;
  int rows, col_div, per_cu;
  double base, half;
  double r[3];  // both operands reduction-contiguous (GATEUP, LINEAR); one (DH, DX); none (DW)
  double e[6];  // by GemmKind; [5]: partial sums
};
const TileCost kLarge = {gmlp::TILE_LARGE, 256, 1, 1, 0.69, 0, {1.443, 1.477, 1.494}, {11.4, 6.1, 19.0, 6.8, 7.1, 12.0}};
const TileCost kWide = {gmlp::TILE_WIDE, 128, 1, 1, 0.74, 0, {0.846, 0.940, 0.983}, {5.7, 2.7, 9.7, 3.3, 3.7, 2.0}};
// (TALL, four wavefronts: fitted the same way to 160 launches, four GEMMs of 40 shapes, standard deviation 7 %; it is the
// fastest unsplit class in 55 of them, by up to 27 %.  bf16, back to back, without and with the class:
// gate/up with biases, G and U kept, at M=1357, K=1160, N=3096 44.1 -> 35.3 us (gelu 44.1 -> 37.5, silu
// without G and U 37.6 -> 28.8), M=1346, K=2264, N=8120 111 -> 106, dH at M=2048, K=2048, N=5632 60 -> 54,
// down at M=5717, K=1640, N=6432 122 -> 110.  Split reductions are left to the smaller classes.)
const TileCost kTall = {gmlp::TILE_TALL, 192, 1, 1, 0.72, 0, {1.101, 1.156, 0}, {9.2, 3.9, 16.2, 0.4, 0, 0}};
const TileCost kMedium = {gmlp::TILE_MEDIUM_FULL, 128, 2, 2, 0.46, 0.30, {0.967, 0.983, 1.094}, {3.4, 0.6, 8.4, 0.2, 2.4, 0.1}};

double launch_us(const TileCost& c, int kind, int64_t tiles, int64_t kt, int splits, double out_elements) {
  const int64_t slots = (int64_t)c.per_cu * num_cu(), wgs = tiles * splits;
  const double f = (double)(wgs % slots) / (double)slots;
  double rounds = (double)(wgs / slots);
  if (f > 0.0)
    rounds += c.half == 0.0 ? c.base + (1.0 - c.base) * f
              : f <= 0.5    ? c.base + c.half * 2.0 * f
                            : c.base + c.half + (1.0 - c.base - c.half) * (2.0 * f - 1.0);
  double us = 3.1 + rounds * ((double)cdiv(kt, splits) * c.r[kind <= LINEAR ? 0 : kind <= DX ? 1 : 2] + c.e[splits > 1 ? 5 : kind]);
  if (splits > 1) us += 4.0 + (double)splits * out_elements * 4.0 / 2.7e6;
  return us;
}

// The classes and splits for a grid of this many tiles of each class (`wide`, `tall` 0: not built).  At
// least 4 reduction tiles per split, at most max_splits splits.
GemmPlan cheapest(int kind, int64_t large, int64_t wide, int64_t tall, int64_t medium, int64_t kt, double out_elements, int64_t max_splits) {
  GemmPlan best = {gmlp::TILE_LARGE, 1, launch_us(kLarge, kind, large, kt, 1, out_elements)};
  auto consider = [&](const TileCost& c, int64_t tiles) {
    const int64_t most = c.tile_class != gmlp::TILE_TALL ? std::max<int64_t>(1, std::min(max_splits, kt / 4)) : 1;
    for (int64_t s = 1; s <= most; ++s) {
      if (s > 1 && cdiv(kt, cdiv(kt, s)) != s) continue;  // rounding up would leave splits empty
      const double us = launch_us(c, kind, tiles, kt, (int)s, out_elements);
      if (us < best.us) best = GemmPlan{c.tile_class, (int)s, us};
    }
  };
  consider(kMedium, medium);
  if (wide > 0) consider(kWide, wide);
  if (tall > 0) consider(kTall, tall);
  return best;
}
int64_t tiles_of(const TileCost& c, int kind, int64_t rows, int64_t cols) {
  return cdiv(rows, c.rows) * cdiv(cols, tile_cols(kind) / c.col_div);
}

// Large tiles with stream-K: behind whole rounds the launches take 0.9 of the sum of their parts
// (eight shapes of 1.25 to 1.5 rounds, where they are up to 8 % ahead of the 128x256 tiles, 5 % behind
// in one).  Grids of less than a round share out everything; inside a step, where their operands are
// still cached and the partial sums' round trip is what is left, they come out a tenth slower than the
// launch alone.
double streamk_us(int kind, int64_t large, int64_t kt, double out_elements) {
  const int64_t cus = num_cu();
  const double pieces = (double)(large % cus) / (double)cus * (double)kt * 1.5;
  if (large < cus) return 1.1 * (pieces + 43.0);
  return 0.9 * (launch_us(kLarge, kind, large / cus * cus, kt, 1, out_elements) + pieces) + 40.0;
}

// A grid of large tiles that ends in a round filled to half or less can run its whole rounds and
// the rest as two launches: cut along the output columns (forward) or the token rows (dH, dX: their
// weight operand is reduction-strided, every other operand row-major in the rows).  Tile columns or
// rows of the first part, or 0.
int64_t whole_rounds(int kind, int64_t rows, int64_t cols) {
  const int64_t tm = cdiv(rows, 256), tn = cdiv(cols, tile_cols(kind)), cus = num_cu();
  const int64_t along = kind <= LINEAR ? tn : tm, across = kind <= LINEAR ? tm : tn;
  const int64_t rounds = tm * tn / cus, tail = tm * tn % cus, whole = rounds * cus / across;
  return rounds >= 1 && tail > 0 && 2 * tail <= cus && whole >= 1 && whole < along ? whole : 0;
}

// The pipelined kernels take any rows, cols and red but need 32-bit byte offsets into the operands,
// padded to whole tiles; anything larger runs on the predicated MEDIUM class.
GemmPlan make_plan(int dtype, int kind, int64_t rows, int64_t cols, int64_t red, bool may_split) {
  if (dtype == GMLP_F32) {
    // (a down projection of at most 64 rows asks for no workspace in float32: its callers rely on that)
    const int64_t tiles = (kind == DX ? 2 : 1) * cdiv(red, 32);
    GemmPlan p = plan_f32(rows, cols, tiles, kind, may_split && (kind != LINEAR || rows > 64) ? kMaxSplits : 1);
    // a chain of reduction tiles on at most one workgroup per CU: both halves of it at once (a tile takes 0.72 us with one
    // chain on a CU, 0.58 with two; below 8 tiles that is about what adding the halves costs)
    if (kind == LINEAR && p.tile_class == gmlp::TILE_F32_64 && p.splits == 1 && tiles >= 8 && cdiv(rows, 64) * cdiv(cols, 64) <= num_cu())
      p.tile_class = gmlp::TILE_F32_HALVES;
    return p;
  }
  auto up = [](int64_t v, int64_t q) { return (v + q - 1) / q * q; };
  // the buffer base sits up to 4 KB below the operand (shared-M0 loads)
  const int64_t limit = ((int64_t)1 << 31) - 4096;
  auto fits = [&](int64_t elements) { return elements * up(red, 64) * 2 < limit; };
  if (!fits(up(rows, 256)) || !fits(up(cols, 256))) return {gmlp::TILE_MEDIUM, 1, 0};
  // (192-row tiles can reach further past the last row than the others: rows that are a multiple of 256)
  auto tall = [&](int64_t r, int64_t c) { return kind != DW && fits(up(r, 192)) ? tiles_of(kTall, kind, r, c) : 0; };
  const int64_t kt = red_tiles_of(kind, red), large = tiles_of(kLarge, kind, rows, cols);
  const double out = (double)rows * (double)cols * (kind == GATEUP ? 2 : 1);
  GemmPlan p = cheapest(kind, large, kind == DW ? 0 : tiles_of(kWide, kind, rows, cols), tall(rows, cols),
                        tiles_of(kMedium, kind, rows, cols), kt, out, may_split ? kMaxSplits : 1);
  if (p.tile_class == gmlp::TILE_LARGE) return p;
  // large tiles whose thin last round is shared out (stream-K) or run by other tiles may still be ahead
  const int64_t cus = num_cu(), whole = whole_rounds(kind, rows, cols);
  double us = p.us;
  if (plan_streamk(dtype, large, kt).tiles > 0) {
    us = streamk_us(kind, large, kt, out);
    // (TALL's estimates differ from its times by 7 %: it has to be ahead by more than that)
    if (p.tile_class == gmlp::TILE_TALL) us *= 0.9;
  } else if (whole > 0) {
    const int64_t r = kind <= LINEAR ? rows : rows - whole * 256, c = kind <= LINEAR ? cols - whole * tile_cols(kind) : cols;
    us = launch_us(kLarge, kind, large / cus * cus, kt, 1, out) +
         cheapest(kind, tiles_of(kLarge, kind, r, c), tiles_of(kWide, kind, r, c), tall(r, c),
                  tiles_of(kMedium, kind, r, c), kt, 0, 1).us;
  }
  return us < p.us ? GemmPlan{gmlp::TILE_LARGE, 1, us} : p;
}

// make_plan takes a few microseconds of estimating, as long as an enqueue: each host thread keeps the
// plans of the last problems it saw (a function of the arguments and the device's compute units only).
GemmPlan plan_gemm(int dtype, int kind, int64_t rows, int64_t cols, int64_t red, bool may_split) {
  struct Entry {
    int64_t key[4] = {-1, -1, -1, -1};
    GemmPlan plan;
  };
  static thread_local Entry cache[64];
  const int64_t key[4] = {rows, cols, red, (((int64_t)num_cu() * 8 + kind) * 4 + dtype) * 2 + (may_split ? 1 : 0)};
  Entry& e = cache[(uint64_t)(rows * 0x9E3779B1 + cols * 0x85EBCA77 + red * 0xC2B2AE3D + key[3] * 0x27D4EB2F) >> 7 & 63];
  if (!std::equal(key, key + 4, e.key)) {
    e.plan = make_plan(dtype, kind, rows, cols, red, may_split);
    std::copy(key, key + 4, e.key);
  }
  return e.plan;
}

// Splits whose partial sums of `out_bytes` each fit a workspace.
int64_t splits_that_fit(size_t workspace_bytes, double out_bytes) {
  const double n = (double)workspace_bytes / out_bytes;
  return n < 1.0 ? 1 : n < (double)kMaxSplits ? (int64_t)n : kMaxSplits;
}

// Weight gradients of float32 modules: all problems in one grid, on one tile class with one number of
// splits; the problems' partial sums follow each other in the workspace.  (workspace_bytes: plan for
// what a workspace of that size can hold.)
GemmPlan plan_dw_group_f32(int count, int64_t Mred, const int64_t* R, const int64_t* C, size_t workspace_bytes = SIZE_MAX) {
  int64_t t128 = 0, t64 = 0;
  double out_bytes = 0;
  for (int i = 0; i < count; ++i) {
    t128 += cdiv(R[i], 128) * cdiv(C[i], 128);
    t64 += cdiv(R[i], 64) * cdiv(C[i], 64);
    out_bytes += (double)R[i] * (double)C[i] * 4.0;
  }
  return plan_f32(t128, t64, cdiv(Mred, 32), 1, out_bytes, splits_that_fit(workspace_bytes, out_bytes), kSplitF32);
}
size_t dw_group_split_bytes(int count, int splits, const int64_t* R, const int64_t* C) {
  size_t n = 0;
  if (splits > 1)
    for (int i = 0; i < count; ++i) n += (size_t)splits * R[i] * C[i] * sizeof(float);
  return n;
}
// Weight gradients of 16-bit modules: LARGE, or MEDIUM_FULL with or without a split reduction, chosen
// for the problems together (their tiles share the rounds of workgroups).
int64_t dw_group_tiles(const TileCost& c, int count, const int64_t* R, const int64_t* C) {
  int64_t n = 0;
  for (int i = 0; i < count; ++i) n += tiles_of(c, DW, R[i], C[i]);
  return n;
}
GemmPlan plan_dw_group(int count, int64_t Mred, const int64_t* R, const int64_t* C, size_t workspace_bytes = SIZE_MAX) {
  double out = 0;
  for (int i = 0; i < count; ++i) out += (double)R[i] * (double)C[i];
  const int64_t large = dw_group_tiles(kLarge, count, R, C), kt = cdiv(Mred, 64);
  GemmPlan p = cheapest(DW, large, 0, 0, dw_group_tiles(kMedium, count, R, C), kt, out, splits_that_fit(workspace_bytes, 4.0 * out));
  const StreamK sk = plan_streamk(GMLP_F16, large, kt, false);
  if (p.tile_class != gmlp::TILE_LARGE && sk.tiles > 0 && sk.ws_bytes <= workspace_bytes) {
    const double us = streamk_us(DW, large, kt, out);
    if (us < p.us) p = GemmPlan{gmlp::TILE_LARGE, 1, us};
  }
  return p;
}

// Estimated time of a GEMM as run_plan launches it (16-bit types, no stream-K).
double planned_us(int kind, int64_t rows, int64_t cols, int64_t red, const GemmPlan& p) {
  const int64_t kt = red_tiles_of(kind, red), whole = whole_rounds(kind, rows, cols);
  if (p.tile_class != gmlp::TILE_LARGE || whole == 0) return p.us;
  const int64_t r = kind <= LINEAR ? rows : rows - whole * 256, c = kind <= LINEAR ? cols - whole * tile_cols(kind) : cols;
  return launch_us(kLarge, kind, tiles_of(kLarge, kind, rows, cols) / num_cu() * num_cu(), kt, 1, 0) +
         plan_gemm(GMLP_F16, kind, r, c, red, false).us;
}
// ... and of grouped weight gradients: a thin last round runs as a launch of its own.
double planned_dw_group_us(int64_t Mred, int64_t large, const GemmPlan& p) {
  const int64_t cus = num_cu(), rounds = large / cus, tail = large % cus, kt = cdiv(Mred, 64);
  if (p.tile_class != gmlp::TILE_LARGE || rounds < 1 || rounds > 4 || tail == 0 || 2 * tail > cus) return p.us;
  return launch_us(kLarge, DW, rounds * cus, kt, 1, 0) + launch_us(kMedium, DW, 4 * tail, kt, 1, 0);
}

size_t split_workspace_bytes(int splits, int64_t rows, int64_t cols, int accumulator_sets = 1) {
  return splits > 1 ? (size_t)splits * accumulator_sets * rows * cols * sizeof(float) : 0;
}

// A GEMM with a split reduction: `launch` leaves `sets` accumulator sets of fp32 partial sums per split
// in the workspace (per split: the first set [rows, cols], then the second), the second stage adds them
// up in split order and runs the unsplit epilogue.
template <typename T, typename Epi, typename Launch>
hipError_t run_split(gmlp::GemmArgs& ga, int splits, int sets, void* workspace, const typename Epi::Args& ea, int64_t rows,
                     int64_t cols, hipStream_t s, Launch&& launch) {
  ga.splits = splits;
  const size_t set = (size_t)rows * cols, acc_stride = sets == 2 ? set : 0;
  const typename gmlp::EpiPartial<T>::Args pa = {(float*)workspace, sets * set, acc_stride, (int)cols};
  if (hipError_t err = launch(ga, pa)) return err;
  return gmlp::launch_splitk_reduce<T, Epi>((const float*)workspace, splits, sets * set, acc_stride, ea, rows, cols, s);
}

// Runs a GEMM as planned.  run(first, count, plan, sk) launches the output columns (forward) or rows
// (dH, dX) [first, first + count); `sk`: the launch's stream-K plan, or null.
template <typename Run>
hipError_t run_plan(int dtype, int kind, int64_t rows, int64_t cols, int64_t red, const void* workspace, size_t workspace_bytes,
                    Run&& run) {
  const int64_t all = kind <= LINEAR ? cols : rows;
  GemmPlan p = plan_gemm(dtype, kind, rows, cols, red, true);
  if (p.splits > 1 && (workspace == nullptr || workspace_bytes < split_workspace_bytes(p.splits, rows, cols, kind == GATEUP ? 2 : 1)))
    p = plan_gemm(dtype, kind, rows, cols, red, false);
  if (p.tile_class == gmlp::TILE_LARGE) {
    // a thin last round behind a long reduction: its tiles are shared out by reduction range
    const StreamK sk = plan_streamk(dtype, tiles_of(kLarge, kind, rows, cols), red_tiles_of(kind, red));
    if (sk.tiles > 0 && workspace != nullptr && workspace_bytes >= sk.ws_bytes) return run(0, all, p, &sk);
    // behind a short one: the whole rounds, then the rest as a problem of its own, for which the planner
    // usually picks smaller tiles (measured on the gate/up GEMM: 1.375 rounds 114 -> 95 us, 5.375
    // rounds 627 -> 611 us, 3.5 rounds 416 -> 407 us)
    const int64_t whole = whole_rounds(kind, rows, cols);
    if (whole > 0) {
      const int64_t first = whole * (kind <= LINEAR ? tile_cols(kind) : 256), rest = all - first;
      if (hipError_t err = run(0, first, p, nullptr)) return err;
      return run(first, rest, plan_gemm(dtype, kind, kind <= LINEAR ? rows : rest, kind <= LINEAR ? rest : cols, red, false),
                 nullptr);
    }
  }
  return run(0, all, p, nullptr);
}

// dX and the weight gradients as one grid.  Behind each other both end in a round that does not fill the
// chip; in one grid the workgroups with the longer tiles come first and the others fill what those leave.
// Estimated by dealing the workgroups out to the CUs in that order, each at what its class takes in a full
// round (and a fifth of it at a perfect deal: CUs that are at different places of their tiles get a larger share
// of the bandwidth each), and taken where that is ahead of the separate launches' estimates: mostly below about
// 4000 rows (4096x4096x14336 and 7431x2208x3296 stay as they are: many rounds, 0.999 to 1.001 of the time
// either way).  Fitted over 116 shapes of 64 to 8192 rows and 128 to 4700 inputs, each on all four pairs of
// classes and separately: backward passes take 0.907 of the time with this choice, 0.898 with the best one, at worst 1.02.
// Both keep the number of splits that they have by themselves, so that the results are the same bit for bit, and
// one launch adds up the partial sums of both; shared-out tiles (stream-K) keep launches of their own.
struct DxDwPlan {
  bool merged = false, dx_first = true;  // dX in the grid
  int x_class = 0, splits = 1;           // ... its tiles
  int dw_splits = 1;                     // ... and of the weight gradients
  int dw_class = -1;                     // the weight gradients' tiles in one grid of their own, or -1: not one grid
  double cover_us = 0;                   // from when the last tiles of the grid with dX start until it ends
};
// When `slots` that take the next workgroup as they get free are through with n0 workgroups of d0 us and then n1 of d1 us.
double makespan_us(int64_t slots, int64_t n0, double d0, int64_t n1, double d1) {
  const int64_t late_slots = n0 % slots;  // these get free a round later than the others
  const double early = (double)(n0 / slots) * d0, late = late_slots ? early + d0 : early;
  const double work = ((double)n0 * d0 + (double)n1 * d1) / (double)slots;
  auto done_by = [&](double t) {
    auto each = [&](double from) { return (int64_t)std::max(0.0, std::floor((t - from) / d1 + 1e-6)); };
    return late_slots * each(late) + (slots - late_slots) * each(early);
  };
  auto end_from = [&](double from) {  // (the last one ends a whole number of d1 after one of the two moments)
    double t = from + std::max(0.0, std::floor((work - from) / d1)) * d1;
    while (done_by(t) < n1) t += d1;
    return t;
  };
  return std::max(late, std::min(end_from(early), end_from(late)));
}
// float32: the estimates of plan_f32, all on the same tiles.
DxDwPlan make_plan_dx_dw_f32(int64_t M, int64_t K, int64_t N, int count, const int64_t* R, const int64_t* C, size_t workspace_bytes) {
  DxDwPlan p;
  const GemmPlan pw = plan_dw_group_f32(count, M, R, C);
  const size_t dw_bytes = dw_group_split_bytes(count, pw.splits, R, C);
  if (dw_bytes > workspace_bytes) return p;
  if (pw.splits == 1) p.dw_class = pw.tile_class;
  GemmPlan px = plan_gemm(GMLP_F32, DX, M, K, N, true);
  if (px.splits > 1 && workspace_bytes < split_workspace_bytes(px.splits, M, K)) px = plan_gemm(GMLP_F32, DX, M, K, N, false);
  const size_t dx_bytes = split_workspace_bytes(px.splits, M, K);
  if (dx_bytes + dw_bytes > workspace_bytes) return p;
  double best = px.us + pw.us;
  const int64_t cus = num_cu(), kx = cdiv(2 * cdiv(N, 32), px.splits), kw = cdiv(cdiv(M, 32), pw.splits);
  for (int64_t b : {128, 64}) {
    const double* r = b == 128 ? kF32R128 : kF32R64;
    const double e = b == 128 ? kF32E128 : kF32E64;
    const int64_t nx = cdiv(M, b) * cdiv(K, b) * px.splits;
    int64_t nw = 0;
    for (int i = 0; i < count; ++i) nw += cdiv(R[i], b) * cdiv(C[i], b) * pw.splits;
    const int64_t per = std::min<int64_t>(cdiv(nx + nw, cus), b == 128 ? 2 : 3);
    const double dx = (double)kx * r[per - 1] + e, dw = (double)kw * r[per - 1] + e;
    const bool dx_first = dx >= dw;
    double us = kF32Launch + (dx_first ? makespan_us(per * cus, nx, dx, nw, dw) : makespan_us(per * cus, nw, dw, nx, dx));
    if (dx_bytes + dw_bytes > 0) us += kSplitF32 + kF32Traffic * (double)(dx_bytes + dw_bytes);
    if (us < best) {
      best = us;
      p.merged = true;
      p.dx_first = dx_first;
      p.x_class = b == 128 ? gmlp::TILE_F32_128 : gmlp::TILE_F32_64;
      p.splits = px.splits;
      p.dw_splits = pw.splits;
      p.cover_us = nx + nw <= per * cus ? std::max(dx, dw) : std::min(dx, dw);
    }
  }
  return p;
}
DxDwPlan make_plan_dx_dw(int dtype, int64_t M, int64_t K, int64_t N, int count, const int64_t* R, const int64_t* C,
                         size_t workspace_bytes) {
  DxDwPlan p;
  for (int i = 0; i < count; ++i)
    if (plan_gemm(dtype, DW, R[i], C[i], M, false).tile_class == gmlp::TILE_MEDIUM) return p;
  const GemmPlan pw = plan_dw_group(count, M, R, C);
  const size_t dw_bytes = dw_group_split_bytes(count, pw.splits, R, C);
  if (dw_bytes > workspace_bytes) return p;
  const int64_t ktx = red_tiles_of(DX, N), ktw = cdiv(M, 64), large = dw_group_tiles(kLarge, count, R, C);
  if (pw.tile_class == gmlp::TILE_LARGE && plan_streamk(dtype, large, ktw, false).tiles > 0) return p;
  const double dw_us = planned_dw_group_us(M, large, pw);
  if (pw.splits == 1 && dw_us == pw.us) p.dw_class = pw.tile_class;
  GemmPlan px = plan_gemm(dtype, DX, M, K, N, true);
  if (px.splits > 1 && workspace_bytes < split_workspace_bytes(px.splits, M, K)) px = plan_gemm(dtype, DX, M, K, N, false);
  const size_t dx_bytes = split_workspace_bytes(px.splits, M, K);
  if (px.tile_class == gmlp::TILE_MEDIUM || dx_bytes + dw_bytes > workspace_bytes) return p;
  if (px.tile_class == gmlp::TILE_LARGE && plan_streamk(dtype, tiles_of(kLarge, DX, M, K), ktx).tiles > 0) return p;
  double best = planned_us(DX, M, K, N, px) + dw_us;
  const int64_t kt = cdiv(ktx, px.splits), kt_dw = cdiv(ktw, pw.splits), cus = num_cu();
  // (the splits' partial sums are written while other workgroups compute, and are read from the cache)
  const double second = dx_bytes + dw_bytes > 0 ? 1.5 + (double)(dx_bytes + dw_bytes) / 1.8e7 : 0.0;
  auto consider = [&](const TileCost& cx, const TileCost& cw) {
    const int64_t slots = cx.per_cu * cus, nx = tiles_of(cx, DX, M, K) * px.splits, nw = dw_group_tiles(cw, count, R, C) * pw.splits;
    double dx = (double)kt * cx.r[1] + cx.e[px.splits > 1 ? 5 : DX], dw = (double)kt_dw * cw.r[2] + cw.e[pw.splits > 1 ? 5 : DW];
    if (nx + nw < slots) {  // (a partly filled round, see launch_us)
      const double f = (double)(nx + nw) / (double)slots;
      const double fill = cx.half == 0.0 ? cx.base + (1.0 - cx.base) * f
                          : f <= 0.5     ? cx.base + cx.half * 2.0 * f
                                         : cx.base + cx.half + (1.0 - cx.base - cx.half) * (2.0 * f - 1.0);
      dx *= fill;
      dw *= fill;
    }
    const bool dx_first = dx >= dw;
    const double makespan = dx_first ? makespan_us(slots, nx, dx, nw, dw) : makespan_us(slots, nw, dw, nx, dx);
    const double us = 7.5 + 0.8 * makespan + 0.2 * ((double)nx * dx + (double)nw * dw) / (double)slots + second;
    if (us < best) {
      best = us;
      p.merged = true;
      p.dx_first = dx_first;
      p.x_class = cx.tile_class;
      p.splits = px.splits;
      p.dw_splits = pw.splits;
      p.cover_us = nx + nw <= slots ? std::max(dx, dw) : std::min(dx, dw);
    }
  };
  consider(kMedium, kMedium);
  if (pw.splits > 1) return p;
  consider(kLarge, kLarge);
  consider(kWide, kLarge);
  // (a 192-row tile can reach further past the last row than the others: see make_plan)
  if (px.splits == 1 && cdiv(M, 192) * 192 * (cdiv(N, 64) * 64) * 2 < ((int64_t)1 << 31) - 4096) consider(kTall, kLarge);
  return p;
}
DxDwPlan plan_dx_dw(int dtype, int64_t M, int64_t K, int64_t N, int count, const int64_t* R, const int64_t* C,
                    size_t workspace_bytes) {
  struct Entry {
    int64_t key[6] = {-1, -1, -1, -1, -1, -1};
    DxDwPlan plan;
  };
  static thread_local Entry cache[32];
  int64_t wide = 0;  // which of the weights: the gradients are [N, K] or [K, N]
  for (int i = 0; i < count; ++i) wide = wide * 2 + (R[i] == K);
  const int64_t key[6] = {M, K, N, ((int64_t)num_cu() * 4 + dtype) * 8 + count, wide, (int64_t)workspace_bytes};
  Entry& e = cache[(uint64_t)(M * 0x9E3779B1 + K * 0x85EBCA77 + N * 0xC2B2AE3D + key[3] * 0x27D4EB2F + wide) >> 7 & 31];
  if (!std::equal(key, key + 6, e.key)) {
    e.plan = dtype == GMLP_F32 ? make_plan_dx_dw_f32(M, K, N, count, R, C, workspace_bytes)
                               : make_plan_dx_dw(dtype, M, K, N, count, R, C, workspace_bytes);
    std::copy(key, key + 6, e.key);
  }
  return e.plan;
}

std::mutex& lds_registry_mutex() {
  static std::mutex m;
  return m;
}
std::vector<gmlp::LdsKernel*>& lds_registry() {
  static std::vector<gmlp::LdsKernel*> v;
  return v;
}

}  // namespace

namespace gmlp {

LdsKernel::LdsKernel(const void* k, int b) : kernel(k), bytes(b), done{} {
  std::lock_guard<std::mutex> lock(lds_registry_mutex());
  lds_registry().push_back(this);
}

hipError_t prepare_lds_kernels() {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  std::lock_guard<std::mutex> lock(lds_registry_mutex());
  for (LdsKernel* k : lds_registry()) {
    if (hipError_t e = hipFuncSetAttribute(k->kernel, hipFuncAttributeMaxDynamicSharedMemorySize, k->bytes)) return e;
    if (dev >= 0 && dev < 64) k->done[dev].store(1, std::memory_order_release);
  }
  return hipSuccess;
}

}  // namespace gmlp

extern "C" {

int gmlp_abi_version(void) { return GMLP_ABI_VERSION; }
const char* gmlp_last_error(void) { return g_err; }

int gmlp_init(void) {
  (void)num_cu();
  if (hipError_t e = gmlp::prepare_lds_kernels()) return hip_result(__func__, e);
  float* scratch = nullptr;
  return hip_result(__func__, gmlp::colsum_static_scratch(&scratch, nullptr));
}

size_t gmlp_workspace_bytes(int op, int64_t M, int64_t K, int64_t N, int dtype) {
  // gmlp_dw_bwd_grouped, any set of problems (the plan depends on all of them together): the most that
  // shared-out tiles can take, a slot per compute unit for them and one for the workgroups.  Split reductions
  // of long batches can take more, see gmlp_dw_bwd_grouped_workspace_bytes.
  if (op == GMLP_OP_DW_BWD_GROUPED) return dtype == GMLP_F32 ? 0 : (size_t)2 * num_cu() * 65536 * sizeof(float);
  if (M < 1 || N < 1) return 0;
  if (op == GMLP_OP_COLSUM) return gmlp::colsum_workspace_bytes(M, N);
  if (K < 1) return 0;
  // Each operation asks for what its plan uses: partial sums of a split reduction, or, large tiles whose
  // grid ends in a thinly filled round, the stream-K slots.
  auto bytes = [&](int kind, int64_t rows, int64_t cols, int64_t red) -> size_t {
    const GemmPlan p = plan_gemm(dtype, kind, rows, cols, red, true);
    if (p.tile_class == gmlp::TILE_LARGE)
      return plan_streamk(dtype, tiles_of(kLarge, kind, rows, cols), red_tiles_of(kind, red)).ws_bytes;
    return split_workspace_bytes(p.splits, rows, cols, kind == GATEUP ? 2 : 1);
  };
  if (op == GMLP_OP_GATEUP_FWD) return bytes(GATEUP, M, N, K);  // gmlp_gateup_fwd(M, K, N)
  if (op == GMLP_OP_LINEAR_FWD) return bytes(LINEAR, M, N, K);  // gmlp_linear_fwd(M, R = K, C = N)
  if (op == GMLP_OP_DX_BWD) return bytes(DX, M, K, N);          // gmlp_dx_bwd(M, K, N): two segments of N
  if (op == GMLP_OP_DH_BWD) return bytes(DH, M, N, K);          // gmlp_dh_bwd(M, K, N)
  // gmlp_dw_bwd(Mred = M, R = K, C = N): out [K,N], reduction over the M token rows
  if (op == GMLP_OP_DW_BWD) return gmlp_dw_bwd_grouped_workspace_bytes(1, M, &K, &N, dtype);
  return 0;
}

int gmlp_gateup_fwd(const void* x, const void* w_gate, const void* w_up, const void* b_gate,
                    const void* b_up, void* h, void* g_save, void* u_save, uint8_t* mask_out,
                    int64_t M, int64_t K, int64_t N, int dtype, int act, float dropout_p,
                    uint64_t seed, uint64_t offset, void* workspace, size_t workspace_bytes,
                    void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(x); GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up); GMLP_REQUIRE_PTR(h);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ACT(act);
  DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(x); GMLP_REQUIRE_ALIGNED(w_gate); GMLP_REQUIRE_ALIGNED(w_up);
  GMLP_REQUIRE_ALIGNED(b_gate); GMLP_REQUIRE_ALIGNED(b_up); GMLP_REQUIRE_ALIGNED(h);
  GMLP_REQUIRE_ALIGNED(g_save); GMLP_REQUIRE_ALIGNED(u_save); GMLP_REQUIRE_ALIGNED(mask_out);
  GMLP_REQUIRE_ALIGNED(workspace);

  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    // The GEMM over output columns [col0, col0 + cols): every per-column pointer moves along, the
    // row pitch of the outputs stays N.
    auto run = [&](int64_t col0, int64_t cols, const GemmPlan& plan, const StreamK* sk) -> hipError_t {
      GemmArgs ga = {};
      ga.nxcd = num_xcd();
      if (sk) use_streamk(*sk, ga, workspace, workspace_bytes);
      ga.A[0] = x; ga.A[1] = x;
      ga.B[0] = (const T*)w_gate + col0 * K; ga.B[1] = (const T*)w_up + col0 * K;
      ga.M = (int)M; ga.N = (int)cols; ga.K = (int)K; ga.lda = (int)K; ga.ldb = (int)K;
      ga.nseg = 1; ga.group_m = pick_group(M, cols, 2); ga.rotate = M <= 512;
      auto at = [&](const void* p) { return p ? (const T*)p + col0 : nullptr; };
      typename EpiGateUp<T>::Args ea = {(T*)at(h), (T*)at(g_save), (T*)at(u_save), mask_out ? mask_out + col0 : nullptr,
                                        at(b_gate), at(b_up), (int)N, act, d, (size_t)col0};
      if (plan.splits > 1)
        return run_split<T, EpiGateUp<T>>(ga, plan.splits, 2, workspace, ea, M, cols, s,
                                          [&](auto& g, auto& pa) { return launch_gateup_split<T>(plan.tile_class, g, pa, s); });
      return launch_gateup<T>(plan.tile_class, ga, ea, s);
    };
    return run_plan(dtype, GATEUP, M, N, K, workspace, workspace_bytes, run);
  });
  return hip_result(__func__, e);
}

int gmlp_linear_fwd(const void* a, const void* w, const void* bias, void* out, int64_t M, int64_t R,
                    int64_t C, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(a); GMLP_REQUIRE_PTR(w); GMLP_REQUIRE_PTR(out);
  GMLP_REQUIRE_DTYPE(dtype);
  if (int rc = check_dims(__func__, M, R, C)) return rc;
  if (int rc = check_mult8(__func__, "R", R)) return rc;
  if (int rc = check_mult8(__func__, "C", C)) return rc;
  GMLP_REQUIRE_ALIGNED(a); GMLP_REQUIRE_ALIGNED(w); GMLP_REQUIRE_ALIGNED(bias);
  GMLP_REQUIRE_ALIGNED(out); GMLP_REQUIRE_ALIGNED(workspace);

  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    // The GEMM over output columns [col0, col0 + cols); the row pitch of `out` stays C.
    auto run = [&](int64_t col0, int64_t cols, const GemmPlan& plan, const StreamK* sk) -> hipError_t {
      GemmArgs ga = {};
      ga.nxcd = num_xcd();
      if (sk) use_streamk(*sk, ga, workspace, workspace_bytes);
      ga.A[0] = a; ga.A[1] = a;
      ga.B[0] = (const T*)w + col0 * R; ga.B[1] = ga.B[0];
      ga.M = (int)M; ga.N = (int)cols; ga.K = (int)R; ga.lda = (int)R; ga.ldb = (int)R;
      ga.nseg = 1; ga.group_m = pick_group(M, cols); ga.rotate = M <= 512;
      typename EpiStore<T>::Args ea = {(T*)out + col0, bias ? (const T*)bias + col0 : nullptr, (int)C};
      if (plan.splits > 1)
        return run_split<T, EpiStore<T>>(ga, plan.splits, 1, workspace, ea, M, cols, s,
                                         [&](auto& g, auto& pa) { return launch_linear_split<T>(plan.tile_class, g, pa, s); });
      return launch_linear<T>(plan.tile_class, ga, ea, s);
    };
    return run_plan(dtype, LINEAR, M, C, R, workspace, workspace_bytes, run);
  });
  return hip_result(__func__, e);
}

int gmlp_dh_bwd(const void* dy, const void* w_down, const void* g, const void* u, void* dg, void* du,
                int64_t M, int64_t K, int64_t N, int dtype, int act, float dropout_p, uint64_t seed,
                uint64_t offset, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(dy); GMLP_REQUIRE_PTR(w_down); GMLP_REQUIRE_PTR(g); GMLP_REQUIRE_PTR(u);
  GMLP_REQUIRE_PTR(dg); GMLP_REQUIRE_PTR(du);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ACT(act);
  DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(dy); GMLP_REQUIRE_ALIGNED(w_down); GMLP_REQUIRE_ALIGNED(g);
  GMLP_REQUIRE_ALIGNED(u); GMLP_REQUIRE_ALIGNED(dg); GMLP_REQUIRE_ALIGNED(du);
  GMLP_REQUIRE_ALIGNED(workspace);

  // dH[M,N] = dY[M,K] · W_down[K,N]: reduction over K; B is reduction-strided ([K,N] row-major).
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    // The GEMM over output rows [row0, row0 + rows): every per-row pointer moves along.
    auto run = [&](int64_t row0, int64_t rows, const GemmPlan& plan, const StreamK* sk) -> hipError_t {
      GemmArgs ga = {};
      ga.nxcd = num_xcd();
      if (sk) use_streamk(*sk, ga, workspace, workspace_bytes);
      ga.A[0] = (const T*)dy + row0 * K; ga.A[1] = ga.A[0]; ga.B[0] = w_down; ga.B[1] = w_down;
      ga.M = (int)rows; ga.N = (int)N; ga.K = (int)K; ga.lda = (int)K; ga.ldb = (int)N;
      ga.nseg = 1; ga.group_m = pick_group(rows, N);
      const size_t e0 = (size_t)row0 * N;
      typename EpiDh<T>::Args ea = {(const T*)g + e0, (const T*)u + e0, (T*)dg + e0, (T*)du + e0, (int)N, act, d, e0};
      if (plan.splits > 1)  // (the partial sums' kernel of dX, with one reduction segment)
        return run_split<T, EpiDh<T>>(ga, plan.splits, 1, workspace, ea, rows, N, s,
                                      [&](auto& g, auto& pa) { return launch_dx_split<T>(plan.tile_class, g, pa, s); });
      return launch_dh<T>(plan.tile_class, ga, ea, s);
    };
    return run_plan(dtype, DH, M, N, K, workspace, workspace_bytes, run);
  });
  return hip_result(__func__, e);
}

int gmlp_gating_bwd(const void* dh, const void* g, const void* u, void* dg, void* du, int64_t M,
                    int64_t N, int dtype, int act, float dropout_p, uint64_t seed, uint64_t offset,
                    void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(dh); GMLP_REQUIRE_PTR(g); GMLP_REQUIRE_PTR(u); GMLP_REQUIRE_PTR(dg);
  GMLP_REQUIRE_PTR(du);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ACT(act);
  DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, 8, N)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(dh); GMLP_REQUIRE_ALIGNED(g); GMLP_REQUIRE_ALIGNED(u);
  GMLP_REQUIRE_ALIGNED(dg); GMLP_REQUIRE_ALIGNED(du);
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) {
    typedef decltype(tag) T;
    return launch_gating_bwd<T>((const T*)dh, (const T*)g, (const T*)u, (T*)dg, (T*)du, M, N, act, d, s);
  });
  return hip_result(__func__, e);
}

int gmlp_dx_bwd(const void* dg, const void* du, const void* w_gate, const void* w_up, void* dx,
                int64_t M, int64_t K, int64_t N, int dtype, void* workspace, size_t workspace_bytes,
                void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(dg); GMLP_REQUIRE_PTR(du); GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up);
  GMLP_REQUIRE_PTR(dx);
  GMLP_REQUIRE_DTYPE(dtype);
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(dg); GMLP_REQUIRE_ALIGNED(du); GMLP_REQUIRE_ALIGNED(w_gate);
  GMLP_REQUIRE_ALIGNED(w_up); GMLP_REQUIRE_ALIGNED(dx); GMLP_REQUIRE_ALIGNED(workspace);

  // dX[M,K] = dG[M,N]·W_gate[N,K] + dU[M,N]·W_up[N,K]: two reduction segments of length N.
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    // The GEMM over output rows [row0, row0 + rows).
    auto run = [&](int64_t row0, int64_t rows, const GemmPlan& plan, const StreamK* sk) -> hipError_t {
      GemmArgs ga = {};
      ga.nxcd = num_xcd();
      if (sk) use_streamk(*sk, ga, workspace, workspace_bytes);
      ga.A[0] = (const T*)dg + row0 * N; ga.A[1] = (const T*)du + row0 * N; ga.B[0] = w_gate; ga.B[1] = w_up;
      ga.M = (int)rows; ga.N = (int)K; ga.K = (int)N; ga.lda = (int)N; ga.ldb = (int)K;
      ga.nseg = 2; ga.group_m = pick_group(rows, K);
      // (no rotated reduction order here: a piece has room for one change of direction, and with
      // two reduction segments that is the step from dG·W_gate to dU·W_up)
      typename EpiStore<T>::Args ea = {(T*)dx + row0 * K, nullptr, (int)K};
      if (plan.splits > 1)
        return run_split<T, EpiStore<T>>(ga, plan.splits, 1, workspace, ea, rows, K, s,
                                         [&](auto& g, auto& pa) { return launch_dx_split<T>(plan.tile_class, g, pa, s); });
      return launch_dx<T>(plan.tile_class, ga, ea, s);
    };
    return run_plan(dtype, DX, M, K, N, workspace, workspace_bytes, run);
  });
  return hip_result(__func__, e);
}

int gmlp_dw_bwd(const void* lhs, const void* rhs, void* dw, int64_t Mred, int64_t R, int64_t C,
                int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(lhs); GMLP_REQUIRE_PTR(rhs); GMLP_REQUIRE_PTR(dw);
  GMLP_REQUIRE_DTYPE(dtype);
  if (int rc = check_dims(__func__, Mred, R, C)) return rc;
  if (int rc = check_mult8(__func__, "R", R)) return rc;
  if (int rc = check_mult8(__func__, "C", C)) return rc;
  GMLP_REQUIRE_ALIGNED(lhs); GMLP_REQUIRE_ALIGNED(rhs); GMLP_REQUIRE_ALIGNED(dw);
  GMLP_REQUIRE_ALIGNED(workspace);

  return gmlp_dw_bwd_grouped(1, &lhs, &rhs, &dw, Mred, &R, &C, dtype, workspace, workspace_bytes, stream);
}

size_t gmlp_dw_bwd_grouped_workspace_bytes(int count, int64_t Mred, const int64_t* R, const int64_t* C, int dtype) {
  using namespace gmlp;
  if (count < 1 || count > GEMM_GROUP_MAX || R == nullptr || C == nullptr || Mred < 1) return 0;
  if (dtype == GMLP_F32) {
    for (int i = 0; i < count; ++i)
      if (R[i] < 1 || C[i] < 1) return 0;
    return dw_group_split_bytes(count, plan_dw_group_f32(count, Mred, R, C).splits, R, C);
  }
  bool pipelined = true;
  for (int i = 0; i < count; ++i) {
    if (R[i] < 1 || C[i] < 1) return 0;
    pipelined = pipelined && plan_gemm(dtype, DW, R[i], C[i], Mred, false).tile_class != TILE_MEDIUM;
  }
  if (!pipelined) {  // separate launches, one after the other
    size_t most = 0;
    for (int i = 0; i < count && count > 1; ++i)
      most = std::max(most, gmlp_dw_bwd_grouped_workspace_bytes(1, Mred, R + i, C + i, dtype));
    return most;
  }
  const GemmPlan p = plan_dw_group(count, Mred, R, C);
  if (p.tile_class != TILE_LARGE) return dw_group_split_bytes(count, p.splits, R, C);
  const StreamK sk = plan_streamk(dtype, dw_group_tiles(kLarge, count, R, C), cdiv(Mred, 64), false);
  return sk.tiles > tiles_of(kLarge, DW, R[count - 1], C[count - 1]) ? 0 : sk.ws_bytes;
}

int gmlp_dw_bwd_grouped(int count, const void* const* lhs, const void* const* rhs, void* const* dw,
                        int64_t Mred, const int64_t* R, const int64_t* C, int dtype, void* workspace,
                        size_t workspace_bytes, void* stream) {
  using namespace gmlp;
  if (count < 1 || count > GEMM_GROUP_MAX)
    return fail(GMLP_EINVAL, "%s: count = %d must be in 1..%d", __func__, count, GEMM_GROUP_MAX);
  GMLP_REQUIRE_PTR(lhs); GMLP_REQUIRE_PTR(rhs); GMLP_REQUIRE_PTR(dw); GMLP_REQUIRE_PTR(R);
  GMLP_REQUIRE_PTR(C);
  GMLP_REQUIRE_DTYPE(dtype);
  // One grid when every problem runs on a pipelined tile class; the class is chosen for the
  // problems together (their tiles share the rounds of workgroups).
  bool pipelined = true;
  for (int i = 0; i < count; ++i) {
    GMLP_REQUIRE_PTR(lhs[i]); GMLP_REQUIRE_PTR(rhs[i]); GMLP_REQUIRE_PTR(dw[i]);
    if (int rc = check_dims(__func__, Mred, R[i], C[i])) return rc;
    if (int rc = check_mult8(__func__, "R", R[i])) return rc;
    if (int rc = check_mult8(__func__, "C", C[i])) return rc;
    GMLP_REQUIRE_ALIGNED(lhs[i]); GMLP_REQUIRE_ALIGNED(rhs[i]); GMLP_REQUIRE_ALIGNED(dw[i]);
    pipelined = pipelined && plan_gemm(dtype, DW, R[i], C[i], Mred, false).tile_class != TILE_MEDIUM;
  }
  hipStream_t s = (hipStream_t)stream;
  auto fill = [&](GemmArgs& ga, int i) {
    ga = GemmArgs{};
    ga.nxcd = num_xcd();
    ga.A[0] = lhs[i]; ga.A[1] = lhs[i]; ga.B[0] = rhs[i]; ga.B[1] = rhs[i];
    ga.M = (int)R[i]; ga.N = (int)C[i]; ga.K = (int)Mred; ga.lda = (int)R[i]; ga.ldb = (int)C[i];
    ga.nseg = 1; ga.group_m = pick_group(R[i], C[i]);
  };
  if (!pipelined && count > 1) {  // each problem on the class that suits it
    for (int i = 0; i < count; ++i)
      if (int rc = gmlp_dw_bwd_grouped(1, lhs + i, rhs + i, dw + i, Mred, R + i, C + i, dtype, workspace, workspace_bytes, stream))
        return rc;
    return GMLP_OK;
  }
  if (!pipelined)
    return hip_result(__func__, by_dtype(dtype, [&](auto tag) {
      typedef decltype(tag) T;
      GemmArgs ga;
      fill(ga, 0);
      const typename EpiStore<T>::Args ea = {(T*)dw[0], nullptr, (int)C[0]};
      return launch_dw<T>(TILE_MEDIUM, ga, ea, s);
    }));
  auto plan_group = [&](size_t bytes) {
    return dtype == GMLP_F32 ? plan_dw_group_f32(count, Mred, R, C, bytes) : plan_dw_group(count, Mred, R, C, bytes);
  };
  GemmPlan plan = plan_group(SIZE_MAX);
  if (plan.splits > 1 && (workspace == nullptr || workspace_bytes < dw_group_split_bytes(count, plan.splits, R, C)))
    plan = plan_group(workspace == nullptr ? 0 : workspace_bytes);
  if (dtype == GMLP_F32 || plan.splits > 1) {
    return hip_result(__func__, by_dtype(dtype, [&](auto tag) -> hipError_t {
      typedef decltype(tag) T;
      GemmGroup<typename EpiStore<T>::Args> grp = {};
      GemmGroup<typename EpiPartial<T>::Args> part = {};
      ReduceGroup<T> sum = {};
      grp.count = part.count = sum.count = count;
      float* ws = (float*)workspace;
      for (int i = 0; i < count; ++i) {
        fill(grp.ga[i], i);
        grp.ga[i].splits = plan.splits;
        grp.ea[i] = {(T*)dw[i], nullptr, (int)C[i]};
        part.ga[i] = grp.ga[i];
        part.ea[i] = {ws, (size_t)R[i] * C[i], 0, (int)C[i]};
        sum.ws[i] = ws;
        sum.out[i] = (T*)dw[i];
        sum.n[i] = (size_t)R[i] * C[i];
        sum.splits[i] = plan.splits;
        ws += (size_t)plan.splits * R[i] * C[i];
      }
      if (plan.splits == 1) return launch_dw_group<T>(plan.tile_class, grp, s);
      if (hipError_t err = launch_dw_group_split<T>(plan.tile_class, part, s)) return err;
      return launch_splitk_reduce_group<T>(sum, s);
    }));
  }
  const int group_class = plan.tile_class;
  const int64_t tiles256 = dw_group_tiles(kLarge, count, R, C);
  // A grid of large tiles that ends in a thinly filled round: the last problem gives up a band of
  // its output (whole tile rows or tile columns, whichever comes closer to the tiles of that last
  // round), which runs as a launch of its own on the tile class that suits it; the rest then makes
  // whole rounds.  Both operands are reduction-strided, so the band is a range of columns of one
  // of them: the pointer moves along the rows and the buffer size is trimmed to match.
  int64_t band_rows = 0, band_cols = 0;  // size of the band, in output rows or columns (one is 0)
  const int last = count - 1;
  // With a long reduction the last round's tiles (the last ones of the last problem) are shared out
  // by reduction range instead (stream-K), if the last problem has that many tiles.
  StreamK sk;
  if (group_class == TILE_LARGE) {
    sk = plan_streamk(dtype, tiles256, cdiv(Mred, 64), false);
    if (sk.tiles > cdiv(R[last], 256) * cdiv(C[last], 256) || workspace == nullptr || workspace_bytes < sk.ws_bytes) sk = StreamK{};
  }
  if (group_class == TILE_LARGE && sk.tiles == 0) {
    const int64_t cus = num_cu(), rounds = tiles256 / cus, tail = tiles256 % cus;
    const int64_t tr = (R[last] + 255) / 256, tc = (C[last] + 255) / 256;
    // (worth it for a few rounds only: measured -7 % at 2 rounds, -1 % and less from 8 rounds on)
    if (rounds >= 1 && rounds <= 4 && tail > 0 && 2 * tail <= cus) {
      const int64_t by_rows = (tail + tc - 1) / tc, by_cols = (tail + tr - 1) / tr;  // tile rows / columns
      const bool rows_fit = by_rows < tr, cols_fit = by_cols < tc;
      if (cols_fit && (!rows_fit || by_cols * tr <= by_rows * tc)) band_cols = C[last] - (tc - by_cols) * 256;
      else if (rows_fit) band_rows = R[last] - (tr - by_rows) * 256;
      const int64_t br = band_rows ? band_rows : R[last], bc = band_cols ? band_cols : C[last];
      if ((band_rows || band_cols) && plan_gemm(dtype, DW, br, bc, Mred, false).tile_class == TILE_MEDIUM) band_rows = band_cols = 0;
    }
  }
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    if constexpr (std::is_same<T, float>::value) {
      return hipErrorInvalidValue;  // not reached: returned above
    } else {
      GemmGroup<typename EpiStore<T>::Args> grp = {};
      grp.count = count;
      for (int i = 0; i < count; ++i) {
        fill(grp.ga[i], i);
        grp.ea[i] = typename EpiStore<T>::Args{(T*)dw[i], nullptr, (int)C[i]};
      }
      grp.ga[last].M -= (int)band_rows;
      grp.ga[last].N -= (int)band_cols;
      use_streamk(sk, grp.ga[last], workspace, workspace_bytes);
      if (hipError_t err = launch_dw_group<T>(group_class, grp, s)) return err;
      if (band_rows == 0 && band_cols == 0) return hipSuccess;
      GemmArgs ga;
      fill(ga, last);
      const int64_t r0 = band_rows ? R[last] - band_rows : 0, c0 = band_cols ? C[last] - band_cols : 0;
      ga.A[0] = ga.A[1] = (const T*)lhs[last] + r0;
      ga.B[0] = ga.B[1] = (const T*)rhs[last] + c0;
      ga.a_trim = (int)(r0 * sizeof(T));
      ga.b_trim = (int)(c0 * sizeof(T));
      ga.M = (int)(R[last] - r0);
      ga.N = (int)(C[last] - c0);
      ga.group_m = pick_group(ga.M, ga.N);
      typename EpiStore<T>::Args ea = {(T*)dw[last] + r0 * C[last] + c0, nullptr, (int)C[last]};
      return launch_dw<T>(plan_gemm(dtype, DW, ga.M, ga.N, Mred, false).tile_class, ga, ea, s);
    }
  });
  return hip_result(__func__, e);
}

int gmlp_colsum(const void* a, void* out, void* workspace, int64_t M, int64_t C, int dtype,
                void* stream) {
  const void* as[1] = {a};
  void* outs[1] = {out};
  return gmlp_colsum_grouped(1, as, outs, workspace, M, &C, dtype, stream);
}

int gmlp_colsum_static(const void* a, void* out, int64_t M, int64_t C, int dtype, void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(a); GMLP_REQUIRE_PTR(out);
  GMLP_REQUIRE_DTYPE(dtype);
  if (int rc = check_dims(__func__, M, 8, C)) return rc;
  if (int rc = check_mult8(__func__, "C", C)) return rc;
  if (C > COLSUM_STATIC_MAX_C)
    return fail(GMLP_ESHAPE, "%s: C = %lld exceeds the %lld columns the library's static scratch array holds "
                "(use gmlp_colsum with a workspace)", __func__, (long long)C, (long long)COLSUM_STATIC_MAX_C);
  GMLP_REQUIRE_ALIGNED(a); GMLP_REQUIRE_ALIGNED(out);
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) {
    typedef decltype(tag) T;
    return launch_colsum_static<T>((const T*)a, (T*)out, M, C, s);
  });
  return hip_result(__func__, e);
}

int gmlp_colsum_grouped(int count, const void* const* a, void* const* out, void* workspace, int64_t M,
                        const int64_t* C, int dtype, void* stream) {
  using namespace gmlp;
  if (count < 1 || count > COLSUM_GROUP_MAX)
    return fail(GMLP_EINVAL, "%s: count = %d must be in 1..%d", __func__, count, COLSUM_GROUP_MAX);
  GMLP_REQUIRE_PTR(a); GMLP_REQUIRE_PTR(out); GMLP_REQUIRE_PTR(C); GMLP_REQUIRE_PTR(workspace);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ALIGNED(workspace);
  for (int i = 0; i < count; ++i) {
    GMLP_REQUIRE_PTR(a[i]); GMLP_REQUIRE_PTR(out[i]);
    if (int rc = check_dims(__func__, M, 8, C[i])) return rc;
    if (int rc = check_mult8(__func__, "C", C[i])) return rc;
    GMLP_REQUIRE_ALIGNED(a[i]); GMLP_REQUIRE_ALIGNED(out[i]);
  }
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) {
    typedef decltype(tag) T;
    ColsumGroup<T> g = {};
    char* ws = (char*)workspace;
    for (int i = 0; i < count; ++i) {
      g.a[i] = (const T*)a[i];
      g.out[i] = (T*)out[i];
      g.ws[i] = (float*)ws;
      g.C[i] = C[i];
      ws += colsum_workspace_bytes(M, C[i]);
    }
    return launch_colsum_group<T>(g, count, M, s);
  });
  return hip_result(__func__, e);
}

}  // extern "C"

namespace {
int run_decode(const char* fn, const void* x, const void* w_gate, const void* w_up, const void* w_down, const void* b_gate,
               const void* b_up, const void* b_down, void* h_scratch, void* y, int64_t M, int64_t K, int64_t N, int dtype, int act,
               void* stream) {
  using namespace gmlp;
  hipStream_t s = (hipStream_t)stream;
  const hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    if constexpr (std::is_same<T, float>::value) return hipErrorInvalidValue;  // the callers refuse it
    else
      return launch_decode<T>((const T*)x, (const T*)w_gate, (const T*)w_up, (const T*)w_down, (const T*)b_gate, (const T*)b_up,
                              (const T*)b_down, (T*)h_scratch, (T*)y, (int)M, (int)K, (int)N, act, s);
  });
  return hip_result(fn, e);
}
}  // namespace

extern "C" {

#define GMLP_DECODE_CHECKS()                                                                                           \
  GMLP_REQUIRE_PTR(x); GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up); GMLP_REQUIRE_PTR(w_down);                     \
  GMLP_REQUIRE_PTR(h_scratch); GMLP_REQUIRE_PTR(y);                                                                    \
  GMLP_REQUIRE_DTYPE(dtype);                                                                                           \
  GMLP_REQUIRE_ACT(act);                                                                                               \
  if (int rc = check_dims(__func__, M, K, N)) return rc;                                                               \
  if (dtype == GMLP_F32) return fail(GMLP_ESHAPE, "%s: float32 is not supported by the skinny-M kernels", __func__)
#define GMLP_DECODE_ALIGNED()                                                                                          \
  GMLP_REQUIRE_ALIGNED(x); GMLP_REQUIRE_ALIGNED(w_gate); GMLP_REQUIRE_ALIGNED(w_up);                                   \
  GMLP_REQUIRE_ALIGNED(w_down); GMLP_REQUIRE_ALIGNED(b_gate); GMLP_REQUIRE_ALIGNED(b_up);                              \
  GMLP_REQUIRE_ALIGNED(b_down); GMLP_REQUIRE_ALIGNED(h_scratch); GMLP_REQUIRE_ALIGNED(y)

int gmlp_decode_fwd(const void* x, const void* w_gate, const void* w_up, const void* w_down,
                    const void* b_gate, const void* b_up, const void* b_down, void* h_scratch,
                    void* y, void* workspace, int64_t M, int64_t K, int64_t N, int dtype, int act,
                    void* stream) {
  (void)workspace;
  GMLP_DECODE_CHECKS();
  if (M > 32 || (M > 16 && (K % 256 != 0 || !gmlp::decode_stream_supported((int)M, (int)K, (int)N))))
    return fail(GMLP_ESHAPE,
                "%s: M = %lld exceeds the skinny-M limit (32 when K and N are multiples of 256, at least 768, "
                "and K*N < 2^30; 16 otherwise)",
                __func__, (long long)M);
  if (K % 32 != 0) return fail(GMLP_ESHAPE, "%s: K = %lld must be a multiple of 32", __func__, (long long)K);
  if (N % 256 != 0) return fail(GMLP_ESHAPE, "%s: N = %lld must be a multiple of 256", __func__, (long long)N);
  GMLP_DECODE_ALIGNED();
  return run_decode(__func__, x, w_gate, w_up, w_down, b_gate, b_up, b_down, h_scratch, y, M, K, N, dtype, act, stream);
}

int gmlp_decode_stream_fwd(const void* x, const void* w_gate, const void* w_up, const void* w_down,
                           const void* b_gate, const void* b_up, const void* b_down, void* h_scratch,
                           void* y, int64_t M, int64_t K, int64_t N, int dtype, int act, void* stream) {
  GMLP_DECODE_CHECKS();
  if (M > 32 || !gmlp::decode_stream_supported((int)M, (int)K, (int)N))
    return fail(GMLP_ESHAPE, "%s: needs M <= 32, K and N multiples of 8 and at least 768, K*N < 2^30 (got %lld, %lld, %lld)", __func__,
                (long long)M, (long long)K, (long long)N);
  GMLP_DECODE_ALIGNED();
  return run_decode(__func__, x, w_gate, w_up, w_down, b_gate, b_up, b_down, h_scratch, y, M, K, N, dtype, act, stream);
}

int gmlp_dropout_mask(uint8_t* mask, int64_t M, int64_t N, float dropout_p, uint64_t seed,
                      uint64_t offset, void* stream) {
  using namespace gmlp;
  GMLP_REQUIRE_PTR(mask);
  DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, 8, N)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(mask);
  return hip_result(__func__, launch_dropout_mask(mask, M, N, d, (hipStream_t)stream));
}


}  // extern "C"

// ---------------------------------------------------------------- whole passes in one call
namespace {

// Whether column sums should run at the end of the grid with dX.  A workgroup there sums all rows of 64 columns, 1.1 ns
// a row and byte of an element, from about when the last tiles start.  Launches of their own, the other two terms,
// stream the arrays at 4 TB/s but have a chain of loads too, half as long.  K=200, N=600, bf16, backward pass with three
// bias gradients, in the grid / apart (us): M=4096 41 / 45, 8192 64 / 70, 16384 112 / 110, 32768 216 / 187, 65536 432 / 385;
// K=256, N=512 16384 79 / 87, 32768 146 / 144; float32 32768 497 / 498, 65536 1046 / 879.  Over 1180 shapes of 1500 to
// 140000 rows and 32 to 2048 inputs, bf16 and float32, this takes 1.005 times what the better form does (at worst
// 1.21), in the grid throughout 1.021 (1.41), apart throughout 1.098.
bool sums_beside_tiles(int64_t M, int nsums, const int64_t* cols, int dtype, double cover_us) {
  const double size = dtype == GMLP_F32 ? 4.0 : 2.0, column = size * (double)M;  // bytes
  double all = 0;
  for (int i = 0; i < nsums; ++i) all += column * (double)cols[i];
  return 1.1e-3 * column <= cover_us + 5.0 + std::max(all / 4e6, 0.6e-3 * column);
}

// The gradients of a pass behind dG and dU, its arguments checked: dX (if wanted), the weight gradients
// lhs[i]^T . rhs[i] and the column sums.  The sums run as workgroups at the end of the grid that computes the
// weight gradients, on CUs that its last round leaves free and without a launch (or two) of their own, see
// sums_beside_tiles; unsplit weight gradients in a single grid without dX take them along too (their tiles take
// about ten times what a sum over the same rows does).  Backward passes with three bias gradients over
// 46 shapes of 75 to 8192 rows: 0.73 of the time of separate launches (without biases 0.84), none above 1.02.
int run_gradients(const char* fn, const void* dg, const void* du, const void* w_gate, const void* w_up, void* dx, int count,
                  const void* const* lhs, const void* const* rhs, void* const* dws, int64_t M, int64_t K, int64_t N, const int64_t* R,
                  const int64_t* C, int nsums, const void* const* sum_in, void* const* sum_out, const int64_t* sum_cols, int dtype,
                  void* workspace, size_t ws_bytes, void* stream) {
  using namespace gmlp;
  DxDwPlan plan;
  if (count > 0 && (dx || nsums > 0))
    plan = plan_dx_dw(dtype, M, K, N, count, R, C, workspace ? ws_bytes : 0);
  const bool dx_inside = dx && plan.merged;
  if (dx_inside && nsums > 0 && !sums_beside_tiles(M, nsums, sum_cols, dtype, plan.cover_us)) {
    if (int rc = run_gradients(fn, dg, du, w_gate, w_up, dx, count, lhs, rhs, dws, M, K, N, R, C, 0, nullptr, nullptr, nullptr, dtype,
                               workspace, ws_bytes, stream))
      return rc;
    return gmlp_colsum_grouped(nsums, sum_in, sum_out, workspace, M, sum_cols, dtype, stream);
  }
  if (dx && !dx_inside)
    if (int rc = gmlp_dx_bwd(dg, du, w_gate, w_up, dx, M, K, N, dtype, workspace, ws_bytes, stream)) return rc;
  if (!dx_inside && (nsums == 0 || plan.dw_class < 0)) {
    if (count > 0)
      if (int rc = gmlp_dw_bwd_grouped(count, lhs, rhs, dws, M, R, C, dtype, workspace, ws_bytes, stream)) return rc;
    return nsums > 0 ? gmlp_colsum_grouped(nsums, sum_in, sum_out, workspace, M, sum_cols, dtype, stream) : GMLP_OK;
  }
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = by_dtype(dtype, [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    ReduceGroup<T> sum = {};
    float* ws = (float*)workspace;
    auto partial = [&](int splits, void* out, int64_t rows, int64_t cols) {  // where the partial sums of an output go
      const typename EpiPartial<T>::Args ea = {ws, (size_t)rows * cols, 0, (int)cols};
      sum.ws[sum.count] = ws;
      sum.out[sum.count] = (T*)out;
      sum.n[sum.count] = (size_t)rows * cols;
      sum.splits[sum.count++] = splits;
      ws += (size_t)splits * rows * cols;
      return ea;
    };
    auto launch = [&](auto grp) -> hipError_t {
      GemmArgs& ga = grp.gx;
      ga.nxcd = num_xcd();
      ga.A[0] = dg; ga.A[1] = du; ga.B[0] = w_gate; ga.B[1] = w_up;
      ga.M = dx_inside ? (int)M : 0; ga.N = (int)K; ga.K = (int)N; ga.lda = (int)N; ga.ldb = (int)K;
      ga.nseg = 2; ga.group_m = pick_group(M, K); ga.splits = plan.splits;
      if constexpr (std::is_same<decltype(grp.ex), typename EpiPartial<T>::Args>::value) grp.ex = partial(plan.splits, dx, M, K);
      else grp.ex = {(T*)dx, nullptr, (int)K};
      grp.w.count = count;
      for (int i = 0; i < count; ++i) {
        GemmArgs& gw = grp.w.ga[i];
        gw.nxcd = num_xcd();
        gw.A[0] = gw.A[1] = lhs[i]; gw.B[0] = gw.B[1] = rhs[i];
        gw.M = (int)R[i]; gw.N = (int)C[i]; gw.K = (int)M; gw.lda = (int)R[i]; gw.ldb = (int)C[i];
        gw.nseg = 1; gw.group_m = pick_group(R[i], C[i]); gw.splits = plan.dw_splits;
        if constexpr (std::is_same<decltype(grp.w), GemmGroup<typename EpiPartial<T>::Args>>::value)
          grp.w.ea[i] = partial(plan.dw_splits, dws[i], R[i], C[i]);
        else grp.w.ea[i] = {(T*)dws[i], nullptr, (int)C[i]};
      }
      grp.nsums = nsums;
      grp.sum_rows = M;
      for (int i = 0; i < nsums; ++i) {
        grp.sums.a[i] = (const T*)sum_in[i];
        grp.sums.out[i] = (T*)sum_out[i];
        grp.sums.C[i] = sum_cols[i];
      }
      const int x_class = dx_inside ? plan.x_class : plan.dw_class;
      hipError_t err;
      if constexpr (std::is_same<T, float>::value) err = launch_dx_dw_kt<T, false>(x_class, grp, plan.dx_first, s);
      else err = N % 64 != 0 ? launch_dx_dw_kt<T, true>(x_class, grp, plan.dx_first, s) : launch_dx_dw_kt<T, false>(x_class, grp, plan.dx_first, s);
      if (err) return err;
      return sum.count > 0 ? launch_splitk_reduce_group<T>(sum, s) : hipSuccess;
    };
    const bool dx_split = dx_inside && plan.splits > 1;
    if (dx_inside && plan.dw_splits > 1)
      return dx_split ? launch(DxDwGroup<T, EpiPartial<T>, EpiPartial<T>>{}) : launch(DxDwGroup<T, EpiStore<T>, EpiPartial<T>>{});
    return dx_split ? launch(DxDwGroup<T, EpiPartial<T>>{}) : launch(DxDwGroup<T, EpiStore<T>>{});
  });
  return hip_result(fn, e);
}

size_t bias_workspace_bytes(int64_t M, int64_t K, int64_t N, bool gate, bool up, bool down) {
  return (gate + up) * gmlp::colsum_workspace_bytes(M, N) + down * gmlp::colsum_workspace_bytes(M, K);
}

}  // namespace

extern "C" {

size_t gmlp_mlp_workspace_bytes(int pass, int64_t M, int64_t K, int64_t N, int dtype) {
  if (M < 1 || K < 1 || N < 1) return 0;
  if (pass == GMLP_PASS_FWD) {
    const size_t a = gmlp_workspace_bytes(GMLP_OP_GATEUP_FWD, M, K, N, dtype);
    const size_t b = gmlp_workspace_bytes(GMLP_OP_LINEAR_FWD, M, N, K, dtype);
    return a > b ? a : b;
  }
  if (pass != GMLP_PASS_BWD) return 0;
  const int64_t R[3] = {N, N, K}, C[3] = {K, K, N};
  return std::max({gmlp_workspace_bytes(GMLP_OP_DH_BWD, M, K, N, dtype), gmlp_workspace_bytes(GMLP_OP_DX_BWD, M, K, N, dtype),
                   gmlp_dw_bwd_grouped_workspace_bytes(3, M, R, C, dtype), bias_workspace_bytes(M, K, N, true, true, true)});
}

// The launches of a pass follow each other on one stream, so one buffer of the largest request serves them all;
// dX and the weight gradients, which may share a grid, have their partial sums side by side.  (Whether they do is not asked
// here: the plan goes by the workspace, and a pass would have it made for two sizes each time.)
size_t gmlp_grads_workspace_bytes(int pass, int grads, int64_t M, int64_t K, int64_t N, int dtype) {
  if ((pass != GMLP_PASS_BWD && pass != GMLP_PASS_HIDDEN_BWD) || M < 1 || K < 1 || N < 1) return 0;
  if (pass == GMLP_PASS_HIDDEN_BWD) grads &= ~(GMLP_GRAD_W_DOWN | GMLP_GRAD_B_DOWN);
  const bool hidden = grads & ~(GMLP_GRAD_W_DOWN | GMLP_GRAD_B_DOWN);
  int64_t R[3], C[3];
  int n = 0;
  for (int w : {GMLP_GRAD_W_GATE, GMLP_GRAD_W_UP})
    if (grads & w) R[n] = N, C[n] = K, ++n;
  if (grads & GMLP_GRAD_W_DOWN) R[n] = K, C[n] = N, ++n;
  const size_t dh = hidden && pass == GMLP_PASS_BWD ? gmlp_workspace_bytes(GMLP_OP_DH_BWD, M, K, N, dtype) : 0;
  const size_t dx = grads & GMLP_GRAD_X ? gmlp_workspace_bytes(GMLP_OP_DX_BWD, M, K, N, dtype) : 0;
  const size_t dw = n > 0 ? gmlp_dw_bwd_grouped_workspace_bytes(n, M, R, C, dtype) : 0;
  return std::max({dh, dx + dw,
                   bias_workspace_bytes(M, K, N, grads & GMLP_GRAD_B_GATE, grads & GMLP_GRAD_B_UP, grads & GMLP_GRAD_B_DOWN)});
}

int gmlp_mlp_fwd(const void* x, const void* w_gate, const void* w_up, const void* w_down, const void* b_gate,
                 const void* b_up, const void* b_down, void* y, void* h, void* g_save, void* u_save, int64_t M,
                 int64_t K, int64_t N, int dtype, int act, float dropout_p, uint64_t seed, uint64_t offset,
                 void* workspace, size_t workspace_bytes, void* stream) {
  GMLP_REQUIRE_PTR(x); GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up); GMLP_REQUIRE_PTR(w_down);
  GMLP_REQUIRE_PTR(y); GMLP_REQUIRE_PTR(h);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ACT(act);
  gmlp::DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  GMLP_REQUIRE_ALIGNED(x); GMLP_REQUIRE_ALIGNED(w_gate); GMLP_REQUIRE_ALIGNED(w_up); GMLP_REQUIRE_ALIGNED(w_down);
  GMLP_REQUIRE_ALIGNED(b_gate); GMLP_REQUIRE_ALIGNED(b_up); GMLP_REQUIRE_ALIGNED(b_down); GMLP_REQUIRE_ALIGNED(y);
  GMLP_REQUIRE_ALIGNED(h); GMLP_REQUIRE_ALIGNED(g_save); GMLP_REQUIRE_ALIGNED(u_save); GMLP_REQUIRE_ALIGNED(workspace);
  // both launches are on `stream`, one after the other: they share the workspace
  if (int rc = gmlp_gateup_fwd(x, w_gate, w_up, b_gate, b_up, h, g_save, u_save, nullptr, M, K, N, dtype, act, dropout_p,
                               seed, offset, workspace, workspace_bytes, stream))
    return rc;
  return gmlp_linear_fwd(h, w_down, b_down, y, M, N, K, dtype, workspace, workspace_bytes, stream);
}

int gmlp_mlp_bwd(const void* dy, const void* x, const void* w_gate, const void* w_up, const void* w_down,
                 const void* g, const void* u, const void* h, void* dg, void* du, void* dx, void* dw_gate,
                 void* dw_up, void* dw_down, void* db_gate, void* db_up, void* db_down, int64_t M, int64_t K,
                 int64_t N, int dtype, int act, float dropout_p, uint64_t seed, uint64_t offset, void* workspace,
                 size_t workspace_bytes, void* stream) {
  GMLP_REQUIRE_PTR(dy);
  GMLP_REQUIRE_DTYPE(dtype);
  GMLP_REQUIRE_ACT(act);
  gmlp::DropoutParams d;
  if (int rc = make_dropout(__func__, dropout_p, seed, offset, &d)) return rc;
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  // what each requested output needs
  const bool hidden = dx || dw_gate || dw_up || db_gate || db_up;  // anything behind dG, dU
  if (hidden) {
    GMLP_REQUIRE_PTR(w_down); GMLP_REQUIRE_PTR(g); GMLP_REQUIRE_PTR(u); GMLP_REQUIRE_PTR(dg); GMLP_REQUIRE_PTR(du);
  }
  if (dx) { GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up); }
  if (dw_gate || dw_up) GMLP_REQUIRE_PTR(x);
  if (dw_down) GMLP_REQUIRE_PTR(h);
  GMLP_REQUIRE_ALIGNED(dy); GMLP_REQUIRE_ALIGNED(x); GMLP_REQUIRE_ALIGNED(w_gate); GMLP_REQUIRE_ALIGNED(w_up);
  GMLP_REQUIRE_ALIGNED(w_down); GMLP_REQUIRE_ALIGNED(g); GMLP_REQUIRE_ALIGNED(u); GMLP_REQUIRE_ALIGNED(h);
  GMLP_REQUIRE_ALIGNED(dg); GMLP_REQUIRE_ALIGNED(du); GMLP_REQUIRE_ALIGNED(dx); GMLP_REQUIRE_ALIGNED(dw_gate);
  GMLP_REQUIRE_ALIGNED(dw_up); GMLP_REQUIRE_ALIGNED(dw_down); GMLP_REQUIRE_ALIGNED(db_gate); GMLP_REQUIRE_ALIGNED(db_up);
  GMLP_REQUIRE_ALIGNED(db_down); GMLP_REQUIRE_ALIGNED(workspace);

  // Every launch gets the caller's buffer and uses what it holds (same results from the plainer form that
  // a smaller one leaves).  Bias gradients cannot do without.
  const size_t ws_bytes = workspace != nullptr ? workspace_bytes : 0;
  const size_t sums = bias_workspace_bytes(M, K, N, db_gate, db_up, db_down);
  if (sums > ws_bytes)
    return fail(GMLP_EINVAL, "%s: bias gradients need a workspace of at least %zu bytes (gmlp_grads_workspace_bytes)",
                __func__, sums);

  const void* lhs[3]; const void* rhs[3]; void* dws[3]; int64_t R[3], C[3];
  int n = 0;
  if (dw_gate) { lhs[n] = dg; rhs[n] = x; dws[n] = dw_gate; R[n] = N; C[n] = K; ++n; }
  if (dw_up) { lhs[n] = du; rhs[n] = x; dws[n] = dw_up; R[n] = N; C[n] = K; ++n; }
  if (dw_down) { lhs[n] = dy; rhs[n] = h; dws[n] = dw_down; R[n] = K; C[n] = N; ++n; }
  const void* cs_in[3]; void* cs_out[3]; int64_t cs_c[3];
  int nb = 0;
  if (db_gate) { cs_in[nb] = dg; cs_out[nb] = db_gate; cs_c[nb] = N; ++nb; }
  if (db_up) { cs_in[nb] = du; cs_out[nb] = db_up; cs_c[nb] = N; ++nb; }
  if (db_down) { cs_in[nb] = dy; cs_out[nb] = db_down; cs_c[nb] = K; ++nb; }

  if (hidden)
    if (int rc = gmlp_dh_bwd(dy, w_down, g, u, dg, du, M, K, N, dtype, act, dropout_p, seed, offset, workspace, ws_bytes, stream))
      return rc;
  // Everything on the caller's stream, one launch after the other.  Running the weight gradients
  // on a second stream next to dX was measured and is not done: two grids that each fill the chip
  // run 2.5 to 4 % slower side by side than one after the other (M=8192, K=4096, N=14336), and where
  // grids under-fill the chip (M=2048, K=2048, N=5632) the two event waits that fork and join the
  // streams cost what the overlap gains.
  return run_gradients(__func__, dg, du, w_gate, w_up, dx, n, lhs, rhs, dws, M, K, N, R, C, nb, cs_in, cs_out, cs_c, dtype,
                       workspace, ws_bytes, stream);
}

int gmlp_hidden_bwd(const void* dh, const void* x, const void* w_gate, const void* w_up, const void* g, const void* u,
                    void* dg, void* du, void* dx, void* dw_gate, void* dw_up, void* db_gate, void* db_up, int64_t M,
                    int64_t K, int64_t N, int dtype, int act, float dropout_p, uint64_t seed, uint64_t offset,
                    void* workspace, size_t workspace_bytes, void* stream) {
  GMLP_REQUIRE_DTYPE(dtype);
  if (int rc = check_dims(__func__, M, K, N)) return rc;
  if (int rc = check_mult8(__func__, "K", K)) return rc;
  if (int rc = check_mult8(__func__, "N", N)) return rc;
  if (dx) { GMLP_REQUIRE_PTR(w_gate); GMLP_REQUIRE_PTR(w_up); }
  if (dw_gate || dw_up) GMLP_REQUIRE_PTR(x);
  GMLP_REQUIRE_ALIGNED(x); GMLP_REQUIRE_ALIGNED(w_gate); GMLP_REQUIRE_ALIGNED(w_up); GMLP_REQUIRE_ALIGNED(dx);
  GMLP_REQUIRE_ALIGNED(dw_gate); GMLP_REQUIRE_ALIGNED(dw_up); GMLP_REQUIRE_ALIGNED(db_gate); GMLP_REQUIRE_ALIGNED(db_up);
  GMLP_REQUIRE_ALIGNED(workspace);
  const size_t ws_bytes = workspace != nullptr ? workspace_bytes : 0;
  const size_t sums = bias_workspace_bytes(M, K, N, db_gate, db_up, false);
  if (sums > ws_bytes)
    return fail(GMLP_EINVAL, "%s: bias gradients need a workspace of at least %zu bytes", __func__, sums);
  if (int rc = gmlp_gating_bwd(dh, g, u, dg, du, M, N, dtype, act, dropout_p, seed, offset, stream)) return rc;

  const void* lhs[2]; const void* rhs[2] = {x, x}; void* dws[2];
  const int64_t R[2] = {N, N}, C[2] = {K, K};
  int n = 0;
  if (dw_gate) { lhs[n] = dg; dws[n] = dw_gate; ++n; }
  if (dw_up) { lhs[n] = du; dws[n] = dw_up; ++n; }
  const void* cs_in[2]; void* cs_out[2];
  int nb = 0;
  if (db_gate) { cs_in[nb] = dg; cs_out[nb] = db_gate; ++nb; }
  if (db_up) { cs_in[nb] = du; cs_out[nb] = db_up; ++nb; }
  return run_gradients(__func__, dg, du, w_gate, w_up, dx, n, lhs, rhs, dws, M, K, N, R, C, nb, cs_in, cs_out, R, dtype,
                       workspace, ws_bytes, stream);
}

}  // extern "C"
