// GEMM dispatch: alignment checks, tile choice, and the element-wise kernel
// used for what no MFMA instantiation takes (fewer than 8 columns in an
// operand row, activations on an NN operand).  Ragged N and K (not multiples
// of 8) run on the MFMA path: the last N % 8 columns go out in at most three
// stores, K not a multiple of 8 runs the instantiations that mask the last
// K-step, and rows off the 16-byte grid (leading dimensions not a multiple of 8,
// misaligned pointers) those that load their tiles through registers.
#include <algorithm>
#include <iterator>

#include "gemm_impl.h"

namespace hxmi {
namespace gemm {
hipError_t launch_fast_f16(int tile, bool nn, int epi, bool out_f32, bool rms, const KArgs& k, hipStream_t s);
hipError_t launch_fast_bf16(int tile, bool nn, int epi, bool out_f32, bool rms, const KArgs& k, hipStream_t s);
hipError_t launch_fast_w8(int tile, int epi, bool out_f32, const KArgs& k, hipStream_t s);
hipError_t launch_fast_ragged(int tile, bool bf16, bool nn, int epi, bool out_f32, const KArgs& k, hipStream_t s);
hipError_t launch_fast_unaligned(int tile, bool bf16, bool nn, int epi, bool out_f32, bool rms, const KArgs& k,
                                 hipStream_t s);

namespace {

struct GArgs {
  const char* A;
  const char* B;
  char* C;
  const char* bias;
  int64_t M, N, K, Nout;
  int64_t lda, ldb, ldc, sA, sB, sC, batch;
  float alpha;
  int nn, epi, out_f32;
  int rms;  // scale each output row by rsqrt(mean(A[m,:]^2) + rms_eps)
  float rms_eps;
  float* rs_out;       // rms: the row scales, written by the column-0 threads
  const float* rs_in;  // !rms: given row scales
};

template <typename T>
__device__ __forceinline__ float ld(const char* p, int64_t i) {
  return (float)((const T*)p)[i];
}

// One thread per output element; fp32 accumulation in k order.
template <typename T>
__global__ __launch_bounds__(256) void gemm_elementwise(GArgs a) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per_batch = a.M * a.Nout;
  if (idx >= per_batch * a.batch) return;
  const int64_t b = idx / per_batch;
  const int64_t r = idx - b * per_batch;
  const int64_t m = r / a.Nout, o = r - m * a.Nout;
  const char* A = a.A + b * a.sA * (int64_t)sizeof(T);
  const char* B = a.B + b * a.sB * (int64_t)sizeof(T);
  // packed gate/up columns for SiLU-mul: output o reads packed columns
  // 32*(o/16) + o%16 (gate) and that + 16 (up)
  const int64_t c0 = (a.epi == EPI_SILU_MUL) ? 32 * (o / 16) + (o % 16) : o;
  const int64_t c1 = c0 + 16;
  float acc0 = 0.f, acc1 = 0.f;
  for (int64_t k = 0; k < a.K; ++k) {
    const float av = ld<T>(A, m * a.lda + k);
    const float b0 = a.nn ? ld<T>(B, k * a.ldb + c0) : ld<T>(B, c0 * a.ldb + k);
    acc0 += av * b0;
    if (a.epi == EPI_SILU_MUL) {
      const float b1 = a.nn ? ld<T>(B, k * a.ldb + c1) : ld<T>(B, c1 * a.ldb + k);
      acc1 += av * b1;
    }
  }
  if (a.rms) {
    float ss = 0.f;
    for (int64_t k = 0; k < a.K; ++k) {
      const float av = ld<T>(A, m * a.lda + k);
      ss += av * av;
    }
    const float r = rsqrtf(ss / (float)a.K + a.rms_eps);
    acc0 *= r;
    acc1 *= r;
    if (a.rs_out && o == 0) a.rs_out[m] = r;
  } else if (a.rs_in) {
    acc0 *= a.rs_in[m];
    acc1 *= a.rs_in[m];
  }
  float v = acc0 * a.alpha;
  if (a.epi == EPI_SILU_MUL) {
    v = silu(v) * (acc1 * a.alpha);
  } else {
    if (a.epi == EPI_BIAS || a.epi == EPI_BIAS_GELU_TANH) v += ld<T>(a.bias, o);
    if (a.epi == EPI_GELU_TANH || a.epi == EPI_BIAS_GELU_TANH) v = gelu_tanh(v);
  }
  if (a.out_f32)
    ((float*)a.C)[b * a.sC + m * a.ldc + o] = v;
  else
    ((T*)a.C)[b * a.sC + m * a.ldc + o] = (T)v;
}

// a knob's value, or dflt when unset
int knob_or(Knob k, int dflt) {
  const int64_t v = knob(k);
  return v == KNOB_UNSET ? dflt : (int)v;
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

}  // namespace
}  // namespace gemm

namespace gemm {
namespace {

// Whether the operands suit the direct-to-LDS loads: 16-byte aligned rows
// within 32-bit buffer offsets.  C may lie anywhere (its 16-byte stores take
// any element address at the same cost).
bool operands_aligned(const GemmProblem& p) {
  const bool i8 = p.dtype == DT_W8A16;
  if (i8 && (p.K % 16 || p.N % 8)) return false;
  if (p.epilogue == EPI_SILU_MUL && p.N % 32) return false;
  if (p.K % 8 && p.rms) return false;  // the RMS prologue sums whole fragments
  if (p.lda % 8 || p.ldb % (i8 ? 16 : 8)) return false;
  if (p.batch > 1 && (p.sA % 8 || p.sB % (i8 ? 16 : 8))) return false;
  if (!aligned(p.A, 16) || !aligned(p.B, 16)) return false;
  if (p.bias && !aligned(p.bias, 8)) return false;
  // 32-bit buffer offsets inside one tile row-panel
  if ((int64_t)256 * p.lda * 2 >= (1ll << 31) || (int64_t)256 * p.ldb * 2 >= (1ll << 31)) return false;
  if (p.M >= (1ll << 31) || p.N >= (1ll << 31) || p.K >= (1ll << 31)) return false;
  if (p.b_nt == 0 && i8) return false;
  return true;
}

// Whether some MFMA instantiation computes p with operands and C at any
// element address: rows of at least 8 elements (the unaligned tiles load a
// row's last chunk as its last 8 elements) and the epilogues it is built for.
bool any_alignment_ok(const GemmProblem& p) {
  if (p.dtype == DT_W8A16 || p.K < 8 || (!p.b_nt && p.N < 8)) return false;
  if (p.epilogue == EPI_SILU_MUL && p.N % 32) return false;
  if (!p.b_nt && p.epilogue != EPI_NONE && p.epilogue != EPI_BIAS) return false;
  if (p.out_f32 && (p.epilogue != EPI_NONE || p.rms || p.dtype != DT_F16)) return false;
  if (p.rms && (!p.b_nt || p.epilogue == EPI_GELU_TANH || p.epilogue == EPI_BIAS_GELU_TANH)) return false;
  return p.M < (1ll << 31) && p.N < (1ll << 31) && p.K < (1ll << 31);
}

}  // namespace
}  // namespace gemm

bool gemm_fast_path_ok(const GemmProblem& p) {
  return gemm::operands_aligned(p) && p.ldc % 8 == 0 && (p.batch <= 1 || p.sC % 8 == 0) && gemm::aligned(p.C, 16);
}

namespace gemm {
namespace {

// The ragged-K and unaligned instantiations: 128x128 once its tiles cover the CUs.
int tile_of_two(const GemmProblem& p) {
  const int64_t t128 = ((p.M + 127) / 128) * ((p.N + 127) / 128) * p.batch;
  return t128 >= 256 ? TILE_128x128 : TILE_64x64;
}

// The tile an override asks for (p.tile, then the knob), or -1: none, or one
// that does not take p's layout.
int forced_tile(const GemmProblem& p) {
  int tile = p.tile >= 0 ? p.tile : knob_or(KNOB_GEMM_TILE, -1);
  if (tile < 0 || tile >= TILE_COUNT || (tile == TILE_128x192_W8 && (!p.b_nt || p.dtype == DT_W8A16))) return -1;
  if ((tile == TILE_I8_128x256 || tile == TILE_I8_64x256) && p.dtype != DT_W8A16) return -1;
  if (p.epilogue == EPI_SILU_MUL && kTiles[tile].BN < 128) tile = TILE_64x128;
  return tile;
}

KArgs make_kargs(const GemmProblem& p, int tile) {
  const TileShape s = kTiles[tile];
  KArgs k{};
  k.A = (const char*)p.A;
  k.B = (const char*)p.B;
  k.C = (char*)p.C;
  k.bias = (const char*)p.bias;
  k.scale = (const char*)p.scale;
  k.M = (int)p.M;
  k.N = (int)p.N;
  k.K = (int)p.K;
  k.lda = p.lda;
  k.ldb = p.ldb;
  k.ldc = p.ldc;
  k.sA = p.sA;
  k.sB = p.sB;
  k.sC = p.sC;
  k.batch = (int)p.batch;
  k.alpha = p.alpha;
  k.tiles_m = (int)((p.M + s.BM - 1) / s.BM);
  k.tiles_n = (int)((p.N + s.BN - 1) / s.BN);
  const int gm = knob_or(KNOB_GROUP_M, 4);
  k.group_m = gm < 1 ? 1 : (gm > k.tiles_m ? k.tiles_m : gm);
  k.k_last = 0;
  k.rms_eps = p.rms_eps;
  k.rs_out = p.rs_out;
  k.rs_in = p.rs_in;
  return k;
}

hipError_t launch_fast(const GemmProblem& p, int tile, const KArgs& k, hipStream_t stream) {
  if ((int64_t)k.tiles_m * k.tiles_n * k.batch >= (1ll << 31)) return hipErrorInvalidValue;
  if (p.K % 8) return launch_fast_ragged(tile, p.dtype == DT_BF16, !p.b_nt, p.epilogue, p.out_f32, k, stream);
  if (p.rms && p.dtype == DT_W8A16) return hipErrorNotSupported;
  if (p.dtype == DT_W8A16) return launch_fast_w8(tile, p.epilogue, p.out_f32, k, stream);
  if (p.dtype == DT_BF16) return launch_fast_bf16(tile, !p.b_nt, p.epilogue, p.out_f32, p.rms != 0, k, stream);
  return launch_fast_f16(tile, !p.b_nt, p.epilogue, p.out_f32, p.rms != 0, k, stream);
}

}  // namespace
}  // namespace gemm

// Tile and K slices of a GEMM: the pair with the least estimated time.  Per
// 64-deep K-step a tile alone on its CU takes `lat` us (few CUs busy: the
// loads' latency and its own MFMAs) and, with every CU busy, `thr` us of its
// CU (memory contention and the power limit slow it; with few busy, `part` of
// that), `epi` us for its epilogue; per_cu workgroups share a CU.  Splitting K
// over s workgroups puts short outputs on more CUs and costs fix-up round
// trips plus the partial tiles' traffic (SplitCost).
//
// Constants fitted to every tile and 1-8 slices on 1780 shapes, 17-4096 rows,
// 256-12288 columns (int8 up to 151936) and K 512-8192, both layouts, plain,
// with the norm and SiLU-mul, each with its weights out of cache and in L2
// (graph replays on MI355X; two thirds of the shapes random).  Over a shape's
// best pair the one taken costs 1.0 % out of cache and 0.4 % in L2, int8 0.8 %
// in both; constants fitted to eight shapes took 2.1 and 0.9 %, int8 2.1 and
// 2.0, on single shapes up to half again.  us, tile by area and K < 4096 never
// split / those constants / these:
//   20 x 80 x 3800 13.8 / 8.4 / 8.4; 64 x 768 x 3072 12.3 / 8.7 / 8.6; 64 x 2048 x 5632 14.6 / 11.5 / 11.3;
//   256 x 896 x 4864 14.4 / 12.0 / 12.0; 700 x 2560 x 2048 16.6 / 14.6 / 14.4;
//   700 x 4096 x 4096 48.0 / 54.4 / 39.5; 1028 x 2048 x 5632 49.6 / 38.6 / 37.7;
//   2000 x 2048 x 5632 64.1 / 62.1 / 52.1; 512 x 2048 x 5632 22.8 / 22.9 / 22.4;
//   150 x 11264 x 2048 31.3 / 30.6 / 22.7.
// int8 weights: 256 x 151936 x 896 100.8 / 90.0 / 89.3; 150 x 151936 x 896 101.3 / 78.6 / 77.9;
//   17 x 1152 x 896 7.3 / 8.3 / 7.3; 100 x 896 x 896 7.6 / 8.5 / 7.6; 400 x 4096 x 4096 32.9 / 33.5 / 28.4.
namespace {

struct TileCost {
  int id, bm, bn, per_cu;
  float lat, thr, epi, part;
};
constexpr TileCost kCosts[] = {
    {TILE_256x256_W8, 256, 256, 1, 0.601f, 1.186f, 5.444f, 0.626f},
    {TILE_256x128_W8, 256, 128, 1, 0.613f, 0.660f, 3.681f, 0.952f},
    {TILE_128x192_W8, 128, 192, 1, 0.537f, 0.462f, 3.253f, 0.359f},
    {TILE_128x128_W8, 128, 128, 2, 0.629f, 0.423f, 1.018f, 0.986f},
    {TILE_64x128, 64, 128, 2, 0.396f, 0.350f, 1.038f, 0.626f},
    {TILE_128x64, 128, 64, 2, 0.330f, 0.284f, 1.307f, 0.948f},
    {TILE_64x64, 64, 64, 2, 0.182f, 0.236f, 0.392f, 1.000f},
};
// int8 B: a tile's waves convert every weight they multiply, so the two tiles
// of one wave row convert each once; two workgroups a CU cover each other's
// first loads and epilogue
constexpr TileCost kCostsI8[] = {
    {TILE_256x256_W8, 256, 256, 1, 1.319f, 1.709f, 3.265f, 0.914f},
    {TILE_I8_128x256, 128, 256, 2, 1.069f, 0.874f, 1.287f, 0.937f},
    {TILE_I8_64x256, 64, 256, 2, 0.600f, 0.647f, 1.346f, 0.660f},
    {TILE_128x128, 128, 128, 2, 0.514f, 0.798f, 1.522f, 1.000f},
    {TILE_64x128, 64, 128, 2, 0.565f, 0.419f, 0.545f, 0.539f},
    {TILE_128x64, 128, 64, 2, 0.239f, 0.463f, 1.034f, 0.826f},
    {TILE_64x64, 64, 64, 2, 0.398f, 0.251f, 0.250f, 0.941f},
};
// us of a split: once, per slice, and per element of the partial tiles (their
// write and read)
struct SplitCost {
  float once, slice, element;
};
constexpr SplitCost kSplit = {0.204f, 0.769f, 1.39e-6f}, kSplitI8 = {0.285f, 0.632f, 1.40e-6f};

struct Plan {
  int tile, splits;
  float us;
};

// (mn: output tiles of one batch entry)
float plan_us(const GemmProblem& p, const TileCost& c, int64_t mn, int splits) {
  const int64_t tiles = mn * p.batch * splits;
  const int slots = 256 * c.per_cu;  // (per_cu: 1 or 2)
  const int64_t full = c.per_cu == 1 ? tiles / 256 : tiles / 512;
  const int rem = (int)(tiles - full * slots), conc = (rem + 255) / 256;
  const float round = std::max(c.lat, c.per_cu * c.thr);
  const float last = rem ? std::max(c.lat, conc * c.thr * (c.part + (1.f - c.part) * (float)rem / (256.f * conc))) : 0.f;
  const float steps = (float)(((uint32_t)((p.K + 63) / 64) + splits - 1) / (uint32_t)splits);
  float t = steps * ((float)full * round + last);
  if (p.dtype == DT_W8A16) {  // (the weights from HBM, and what of the rest they do not cover)
    const float hbm = (float)(p.N * p.K) * (1.f / 4.04e6f);
    t = std::max(t, hbm) + 0.058f * std::min(t, hbm);
  }
  // an RMSNorm-folded GEMM sums the squares of its A rows in every tile of a
  // row, so narrow tiles repeat that work more often
  if (p.rms) t *= c.bn == 64 ? 1.090f : 0.915f;
  t += 2.6f + c.epi * ((float)full * c.per_cu + conc);
  if (splits > 1) {
    const SplitCost& f = p.dtype == DT_W8A16 ? kSplitI8 : kSplit;
    t += f.once + f.slice * splits + (float)tiles * (float)(c.bm * c.bn) * f.element;
  }
  return t;
}

// (splits > 0: that many slices; otherwise as many as pay)
Plan gemm_plan(const GemmProblem& p, int splits) {
  Plan best{TILE_64x64, 1, 1e30f};
  const bool i8 = p.dtype == DT_W8A16;
  static_assert(std::size(kCosts) == std::size(kCostsI8), "one loop over either");
  for (const TileCost* e = i8 ? kCostsI8 : kCosts, *const end = e + std::size(kCosts); e != end; ++e) {
    const TileCost& c = *e;
    if (c.bn == 64 && p.epilogue == EPI_SILU_MUL) continue;
    if (c.id == TILE_128x192_W8 && !p.b_nt) continue;  // (k-contiguous weights only)
    const int64_t tiles = ((p.M + c.bm - 1) / c.bm) * ((p.N + c.bn - 1) / c.bn);
    const int first = splits > 0 ? splits : 1;
    // slices of at least four K-steps that stay within two rounds of the
    // CUs, their partial tiles within 32 MiB
    const int64_t most = splits > 0    ? splits
                         : tiles > 256 ? 1
                                       : std::min<int64_t>({8, p.K / 256, 512 / tiles,
                                                            ((32 << 20) - kWsCounterBytes) / (tiles * c.bm * c.bn * 4)});
    for (int s = first; s == first || s <= most; s += s < 4 ? 1 : 2) {
      const float us = plan_us(p, c, tiles, s) * (s > 1 ? 1.02f : 1.f);  // (a split has to gain 2 %)
      if (us < best.us) best = {c.id, s, us};
    }
  }
  // 64x64 tiles with a CU each: a fourth LDS stage.  With the weights out of
  // cache, 12-20 K-steps a slice run 4-6 % shorter with it (NN 3-5 %, under
  // the norm's sums 0-1 %), 32 13-15 % (NN 7 %); with everything in L2 up to
  // 20 run 2 % longer, which NN products and the norm are spared (NN 1024^3
  // 6.4 us, 6.5 with it); two tiles a CU 1-4 % longer either way.
  const int64_t t64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch * best.splits;
  if (best.tile == TILE_64x64 && !i8 && t64 <= 256 && p.K >= (p.rms ? 1536 : p.b_nt ? 768 : 1280))
    best.tile = TILE_64x64_S4;
  return best;
}

bool may_split(const GemmProblem& p) {
  // The library's own scratch serves one call of a GPU at a time.  Callers on
  // several streams only order the products that have always used it: those
  // of a long K into few tiles, and forced splits.
  if (p.lib_scratch && (knob(KNOB_SPLITK) != KNOB_UNSET
                            ? p.K < 2048
                            : p.K < 4096 || ((p.M + 63) / 64) * ((p.N + 127) / 128) >= 384))
    return false;
  return p.batch == 1 && !p.out_f32 && !p.rms && p.K >= 512 && p.K % 8 == 0 && gemm_fast_path_ok(p);
}

}  // namespace

int gemm_pick_tile(const GemmProblem& p) {
  if (p.K % 8) return gemm::tile_of_two(p);
  const int forced = gemm::forced_tile(p);
  if (forced >= 0) return forced;
  return gemm_plan(p, 1).tile;
}

// The split-K launch of p: K slices of kc (a multiple of the 64-deep K-step)
// as a batch of GEMMs into the same output (sC = 0), the tile they run and
// the fix-up workspace they need.  False when p does not split; where the
// plan was to run it whole, `whole` receives the tile (gemm_pick_tile's).
static bool split_plan(const GemmProblem& p, GemmProblem& q, int& tile, int64_t& need, int& whole) {
  if (!may_split(p)) return false;
  const int64_t want = knob(KNOB_SPLITK);
  const Plan plan =
      gemm_plan(p, want == KNOB_UNSET ? 0 : (int)std::max<int64_t>(1, std::min<int64_t>(16, want)));
  const int splits = plan.splits;
  tile = gemm::forced_tile(p);
  if (tile < 0) tile = plan.tile;
  if (splits <= 1) {
    whole = tile;
    return false;
  }
  q = p;
  const int64_t kc = ((p.K + splits - 1) / splits + 63) / 64 * 64;
  q.K = kc;
  q.batch = (p.K + kc - 1) / kc;
  q.sA = kc;
  q.sB = p.b_nt ? kc : kc * p.ldb;
  q.sC = 0;
  const gemm::TileShape s = gemm::kTiles[tile];
  const int64_t tiles = ((p.M + s.BM - 1) / s.BM) * ((p.N + s.BN - 1) / s.BN);
  need = kWsCounterBytes + tiles * q.batch * s.BM * s.BN * 4;
  return q.batch > 1 && tiles <= kWsMaxTiles;
}

int64_t gemm_workspace_bytes(const GemmProblem& p) {
  GemmProblem q;
  int tile, whole;
  int64_t need;
  return split_plan(p, q, tile, need, whole) ? need : 0;
}

hipError_t launch_gemm(const GemmProblem& p, hipStream_t stream) {
  if (p.M == 0 || p.N == 0 || p.batch == 0) return hipSuccess;
  const bool i8 = p.dtype == DT_W8A16;
  if (!gemm_fast_path_ok(p)) {
    if (i8) return hipErrorNotSupported;
    if (gemm::any_alignment_ok(p)) {
      if (gemm::operands_aligned(p)) {  // only C is off the 16-byte grid
        const int tile = gemm_pick_tile(p);
        return gemm::launch_fast(p, tile, gemm::make_kargs(p, tile), stream);
      }
      const int tile = gemm::tile_of_two(p);
      const gemm::KArgs k = gemm::make_kargs(p, tile);
      if ((int64_t)k.tiles_m * k.tiles_n * k.batch >= (1ll << 31)) return hipErrorInvalidValue;
      return gemm::launch_fast_unaligned(tile, p.dtype == DT_BF16, !p.b_nt, p.epilogue, p.out_f32, p.rms != 0, k,
                                         stream);
    }
    gemm::GArgs g;
    g.A = (const char*)p.A;
    g.B = (const char*)p.B;
    g.C = (char*)p.C;
    g.bias = (const char*)p.bias;
    g.M = p.M;
    g.N = p.N;
    g.K = p.K;
    g.Nout = p.epilogue == EPI_SILU_MUL ? p.N / 2 : p.N;
    g.lda = p.lda;
    g.ldb = p.ldb;
    g.ldc = p.ldc;
    g.sA = p.sA;
    g.sB = p.sB;
    g.sC = p.sC;
    g.batch = p.batch;
    g.alpha = p.alpha;
    g.nn = !p.b_nt;
    g.epi = p.epilogue;
    g.out_f32 = p.out_f32;
    g.rms = p.rms;
    g.rms_eps = p.rms_eps;
    g.rs_out = p.rs_out;
    g.rs_in = p.rs_in;
    const int64_t total = p.batch * p.M * g.Nout;
    const int64_t blocks = (total + 255) / 256;
    if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
    if (p.dtype == DT_BF16)
      hipLaunchKernelGGL(gemm::gemm_elementwise<__bf16>, dim3((unsigned)blocks), dim3(256), 0, stream, g);
    else
      hipLaunchKernelGGL(gemm::gemm_elementwise<_Float16>, dim3((unsigned)blocks), dim3(256), 0, stream, g);
    return hipGetLastError();
  }

  GemmProblem q;
  int tile, whole = -1;
  int64_t need;
  if (p.ws && split_plan(p, q, tile, need, whole) && p.ws_bytes >= need && ((uintptr_t)p.ws % 256) == 0) {
    // K slices as a batch into one output; the last slice to finish a tile
    // adds the fp32 partials (in the workspace) and runs the epilogue
    gemm::KArgs k = gemm::make_kargs(q, tile);
    k.k_last = (int)(p.K - (q.batch - 1) * q.K);
    k.fix = (char*)p.ws;
    return gemm::launch_fast(q, tile, k, stream);
  }

  if (whole < 0) whole = gemm_pick_tile(p);
  return gemm::launch_fast(p, whole, gemm::make_kargs(p, whole), stream);
}

GemmProblem w8a16_as_gemm(const GemvProblem& p) {
  GemmProblem q{};
  q.A = p.x;
  q.B = p.W;
  q.C = p.y;
  q.bias = p.bias;
  q.scale = p.scale;
  q.M = p.M;
  q.N = p.N;
  q.K = p.K;
  q.lda = p.ldx;
  q.ldb = p.ldw;
  q.ldc = p.ldy;
  q.batch = 1;
  q.alpha = 1.f;
  q.dtype = DT_W8A16;
  q.b_nt = 1;
  q.epilogue = p.bias ? EPI_BIAS : EPI_NONE;
  q.tile = gemm::knob_or(KNOB_W8_TILE, -1);
  return q;
}

hipError_t launch_w8a16_gemm(const GemvProblem& p, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return hipSuccess;
  GemmProblem q = w8a16_as_gemm(p);
  q.ws = ws;
  q.ws_bytes = ws_bytes;
  if (!gemm_fast_path_ok(q) || ((uintptr_t)p.scale % 8) != 0) return hipErrorNotSupported;
  return launch_gemm(q, stream);
}

}  // namespace hxmi
