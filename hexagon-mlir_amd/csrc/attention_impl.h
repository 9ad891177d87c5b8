// Fused attention O = softmax(scale * Q.K^T + mask) . V in fp16 or bf16 for
// head dims that are multiples of 8 up to 128, with an optional additive fp16
// mask, a causal rule and grouped K/V heads.
//
// The reference lowers tm_tensor.attention to batch_matmul(Q, K^T), a scale,
// the mask add, a row softmax and batch_matmul(P, V) (LowerTmTensor.cpp:91-250,
// mask at :158-163), each a separate pass over HBM.  Here one kernel streams
// K and V once per query block and keeps S and P in registers (online
// softmax, Milakov & Gimelshein 2018, the blockwise form the reference's
// test/python/triton/test_online_softmax.py:30-81 exercises):
//   * a workgroup owns QG x 32 queries of one (batch, head) slice and runs
//     QG x KS waves: wave (qg, kh) takes the 32 queries of group qg against
//     every KS-th block of 32 keys, and the KS partial (max, sum, O) of a
//     query group are merged through LDS at the end;
//   * K and V pass through two LDS stages of 128 keys (D = 64; 64 keys for
//     D = 128) with direct global->LDS buffer loads, one stage ahead of the
//     one computed; rows out of range read as zeros, and a head dim below
//     64 / 128 fills its rows up with zeros (72-96 leave out the MFMAs of the
//     last quarter);
//   * S is computed as D[key][query] = K . Q^T with v_mfma_f32_32x32x16_f16,
//     so every lane owns one query's scores: the row max / sum are in-lane
//     plus one exchange with the lane 32 away;
//   * the running max is only raised when a block's max exceeds it by more
//     than 8 (in log2 units), so most blocks skip the rescale of O; the
//     unnormalised weights then stay below 2^8, well inside fp16;
//   * the 16-bit probabilities of a 32-key block are exactly the B operand of
//     the P.V MFMA for two 16-key steps (the k order inside an MFMA is free as
//     long as both operands use the same one); the matching V^T operand comes
//     from LDS with ds_read_b64_tr_b16, so P never leaves registers;
//   * the vector ALUs bound it (a 32 x 32 tile's softmax is ~62 of their
//     instructions, 16 of them v_exp_f32 at half rate, against 8-16 MFMAs of 32
//     clocks).  Two blocks at a time share one maximum, one rescale test and
//     two independent MFMA chains, and leave four waves a SIMD at head dim
//     64 (122 registers); with the stage loads out of the way, 32 heads x
//     2048 x 2048 at head dim 64 went 53.0 -> 42.9 us (800 TFLOP/s), causal
//     33.2 -> 26.3, head dim 128 x 4096 312 -> 277 us (994 TFLOP/s) against one
//     stage of twice the keys, waited for whole, and one block at a time;
//   * mask entries are read one stage ahead, 32 contiguous bytes a lane
//     wherever the rows start; loaded as a stage began, 8 bytes (rows off the
//     8-byte grid: 2) at a time, they took longer than the rest of the kernel
//     (32 x 1024 x 1024, D 64: 31.9 -> 20.8 us, causal 22.0 -> 15.5, unmasked
//     14.0 and 11.4; 64 x 1000, D 128 causal 72.6 -> 35.9, unmasked 27);
//   * O = D[d][query] accumulates in registers and is divided by the sum of
//     the same 16-bit weights once at the end.  A query whose every key is
//     masked divides 0 by 0 (NaN), as the reference's decomposition does.
#pragma once

#include <type_traits>

#include "hxmi_common.h"
#include "hxmi_internal.h"

namespace hxmi {
namespace attn {

constexpr float kLog2e = 1.4426950408889634f;

enum OrderId { ORDER_SLICES = 0, ORDER_HEAVY, ORDER_PAIRED };

struct AArgs {
  const char* q;
  const char* k;
  const char* v;
  char* o;
  const char* mask;
  int bh, sq, skv, d;
  int nqb;         // query blocks per slice
  int kv_group;    // query slices per K/V slice
  int mask_group;  // query slices per mask slice
  int causal_off;  // key > query + causal_off is masked (skv: no causal rule)
  int order;       // OrderId: workgroup -> (slice, query block)
  int64_t ldq, ldk, ldv, ldo, ldm;  // row strides, elements
  int64_t bq, bk, bv, bo, bm;       // slice strides, elements
  float c;                          // scale * log2(e)
};

// Combine a value with the one of the lane 32 away (v_permlane32_swap: one
// VALU op instead of a round trip through LDS).
__device__ __forceinline__ float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Workgroup -> (slice, query block).  Workgroups go round-robin over the 8
// XCDs; each XCD takes a contiguous run of slices, so the query blocks of a
// slice (and slices sharing a K/V head) read K and V through one L2.
//
// Under the causal rule a query block's work grows with its index, and the
// slices' blocks in index order put blocks of like weight on one CU (2048
// queries, 32 slices, 16 blocks each: the CU that holds two last blocks did
// 1.9 times the mean).  The heaviest blocks of all slices go first instead
// (ORDER_HEAVY).  When every workgroup is resident at once, two to a CU, the
// first 256 take one CU each and the rest join them: those run from the
// lightest up (ORDER_PAIRED), so each CU holds a heavy and a light block.
__device__ __forceinline__ void map_block(int id, const AArgs& a, int& bh, int& qb) {
  const int total = a.bh * a.nqb;
  if (a.order == ORDER_SLICES) {
    const int per = total >> 3, rem = total & 7, xcd = id & 7;
    const int r = xcd * per + (xcd < rem ? xcd : rem) + (id >> 3);
    bh = r / a.nqb;
    qb = r - bh * a.nqb;
    return;
  }
  // whole slices per XCD when they divide; else over all (xcd 0)
  const int xs = (a.bh & 7) ? 0 : 3;
  const int hx = a.bh >> xs, x = id & ((1 << xs) - 1);
  int j = id >> xs;
  const int first = 256 >> xs;
  if (a.order == ORDER_PAIRED && j >= first) j = first + (total >> xs) - 1 - j;
  const int t = j / hx;
  bh = x * hx + j - t * hx;
  qb = a.nqb - 1 - t;
}

// The 16-bit type's MFMA, two weights rounded to it, and c plus their sum.
template <typename T>
struct Num;
template <>
struct Num<_Float16> {
  typedef half2v pair;
  static __device__ __forceinline__ float16v mfma(short8v a, short8v b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8v, a), __builtin_bit_cast(half8v, b), c, 0,
                                                  0, 0);
  }
  static __device__ __forceinline__ float add_pair(pair p, float c) {
    return __builtin_amdgcn_fdot2(p, half2v{(_Float16)1.0f, (_Float16)1.0f}, c, false);
  }
};
template <>
struct Num<__bf16> {
  typedef bf16x2v pair;
  static __device__ __forceinline__ float16v mfma(short8v a, short8v b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c,
                                                   0, 0, 0);
  }
  static __device__ __forceinline__ float add_pair(pair p, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(p, bf16x2v{(__bf16)1.0f, (__bf16)1.0f}, c, false);
  }
};

// K chunk: [KC][D] fp16, rows of 2*D bytes, 16-byte chunks XOR-swizzled as
// the GEMM's k-contiguous tiles; V chunk: [KC][D], 16-byte chunks XOR-ed with
// a multiple of (key & 3) chosen so the 8 row segments (2 lane groups x 4
// keys x 32 bytes) of one transposing read phase cover all 64 banks.  Both
// are involutions on the chunk index, so the loader inverts them the same way.
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  constexpr int RB = 2 * D;
  return (r / (256 / RB)) & (RB / 16 - 1);
}
template <int D>
__device__ __forceinline__ int v_swz(int r) {
  return (r & 3) << (D == 64 ? 1 : 2);  // 32-byte steps for 128-byte rows, 64-byte for 256
}
template <int D>
__device__ __forceinline__ int k_off(int r, int c) {
  return r * (2 * D) + ((c ^ k_swz<D>(r)) << 4);
}
template <int D>
__device__ __forceinline__ int v_off(int r, int c) {
  return r * (2 * D) + ((c ^ v_swz<D>(r)) << 4);
}

// Head dims up to 64 run in LDS rows of D = 64, others in rows of 128.  K and
// V pass through ST LDS stages of KC keys, 64 KB in all (two workgroups a
// CU); a wave takes NB 32-key blocks at a time (a group), GPC groups a stage.
// DEEP: two stages also where one fills 64 KB (one workgroup a CU).
template <int D, int QG, int KS, bool MASK, bool DEEP>
struct AttnShape {
  static constexpr int NT = 64 * QG * KS;
  static constexpr int KC = D == 64 || KS == 4 ? 128 : 64;
  static constexpr int ST = KC * D > 8192 && !DEEP ? 1 : 2;
  static constexpr int NB = KC / 32 / KS >= 2 && !MASK ? 2 : 1;  // (two blocks' mask entries would not fit)
  static constexpr int GPC = KC / 32 / KS / NB;
  static constexpr int CHUNK = KC * 2 * D;    // bytes of K (and of V) per stage: 16 or 32 KB
  static constexpr int NV = D / 32 * 16 + 2;  // floats per lane in the key-split merge
  static constexpr int WPE = QG * KS / (DEEP ? 4 : 2);  // waves per SIMD that one / two workgroups a CU make
  static constexpr bool ok = NT <= 1024 && (KS - 1) * QG * NV * 64 * 4 <= 2 * ST * CHUNK;
};

typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef int int4u __attribute__((ext_vector_type(4), aligned(2)));  // (mask rows start anywhere)
struct MaskBlock {
  int4v v[2];
};

// DT: 32-wide output tiles computed (fewer than D / 32 for head dims 72-96).
// PART: the head dim a.d is below D; rows fill up with zeros.
template <typename T, int D, int DT, bool PART, int QG, int KS, bool MASK, bool DEEP>
__global__ __launch_bounds__(64 * QG * KS, (AttnShape<D, QG, KS, MASK, DEEP>::WPE)) void attention_fwd(AArgs a) {
  using Sh = AttnShape<D, QG, KS, MASK, DEEP>;
  static_assert(Sh::ok, "attention shape");
  constexpr int NW = QG * KS;
  constexpr int KC = Sh::KC, NB = Sh::NB, GPC = Sh::GPC, ST = Sh::ST;
  constexpr int CHUNK = Sh::CHUNK;
  constexpr int RB = 2 * D;     // bytes per K / V row
  constexpr int DS = DT * 2;    // 16-deep MFMA steps over the head dim
  static_assert(PART || DT == D / 32, "whole rows");
  constexpr int LPW = CHUNK / 1024 / NW;  // 1 KB direct loads of K (and of V) per wave per stage
  static_assert(LPW * NW * 1024 == CHUNK, "stage split");
  __shared__ __attribute__((aligned(1024))) char lds[2 * ST * CHUNK];  // K, V of stage 0, then of stage 1

  const int lane = threadIdx.x & 63;
  // wave-uniform values live in scalar registers, so branches on them are
  // scalar branches rather than exec-masked paths
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qg = w % QG, kh = w / QG;
  const int h = lane >> 5;

  int bh, qb;
  map_block(blockIdx.x, a, bh, qb);
  const int qb0 = qb * (32 * QG);
  const int q0 = qb0 + qg * 32;
  const int qme = q0 + (lane & 31);
  const int kvbh = bh / a.kv_group;
  const char* Q = a.q + (int64_t)bh * a.bq * 2;
  const char* Kp = a.k + (int64_t)kvbh * a.bk * 2;
  const char* Vp = a.v + (int64_t)kvbh * a.bv * 2;

  // keys this workgroup / this wave needs (the causal rule cuts both)
  const int wg_qlast = min(qb0 + 32 * QG, a.sq) - 1;
  const int kend = min(a.skv, wg_qlast + a.causal_off + 1);
  const int wkend = q0 < a.sq ? max(0, min(a.skv, min(q0 + 31, a.sq - 1) + a.causal_off + 1)) : 0;
  const int nchunk = kend > 0 ? (kend + KC - 1) / KC : 0;

  // this lane's mask row (queries past the sequence read the last one's)
  const _Float16* mrow = nullptr;
  if constexpr (MASK)
    mrow = (const _Float16*)a.mask + ((int64_t)(bh / a.mask_group) * a.bm + (int64_t)min(qme, a.sq - 1) * a.ldm);

  // Q fragments of this wave's 32 queries (zero past the sequence).  The
  // loads take no branch (an offset past the buffer reads zeros).  The buffer
  // starts at the wave's first row, so its 32-bit offsets span 32 rows (the
  // host checks those) and a slice may be of any length.
  short8v qf[DS];
  {
    const int left = min(32, a.sq - q0), r = lane & 31;
    const __amdgpu_buffer_rsrc_t rQ =
        make_rsrc(Q + (int64_t)q0 * a.ldq * 2, left > 0 ? (uint32_t)(((left - 1) * a.ldq + a.d) * 2) : 0u);
    const uint32_t row = (uint32_t)r * (uint32_t)a.ldq + h * 8;
#pragma unroll
    for (int s = 0; s < DS; ++s)
      qf[s] = __builtin_bit_cast(
          short8v, load16(rQ, r < left && !(PART && s * 16 + h * 8 >= a.d) ? (row + s * 16) * 2 : kOOB));
  }

  // Direct loads: wave w's load i fills LDS bytes [(i*NW + w) KB, +1 KB) of
  // the stage's K (V); lane l's 16 bytes there are row (i*NW + w) *
  // (1024/RB) + lr, stored chunk cs, which holds the row's chunk cs ^
  // swizzle(row).  The offsets are those of the first stage; a later one
  // moves the buffer's base, and keys from kend on lie past its end.
  const int lr = lane / (RB / 16), cs = lane % (RB / 16);
  uint32_t ko[LPW], vo[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int row = (i * NW + w) * (1024 / RB) + lr;
    const int kc = cs ^ k_swz<D>(row), vc = cs ^ v_swz<D>(row);
    const int64_t kr = row * a.ldk * 2, vr = row * a.ldv * 2;  // (a slice spans at most 2 GiB)
    ko[i] = (PART && kc * 8 >= a.d) || kr >= kOOB ? kOOB : (uint32_t)kr + (kc << 4);
    vo[i] = (PART && vc * 8 >= a.d) || vr >= kOOB ? kOOB : (uint32_t)vr + (vc << 4);
  }
  auto issue = [&](int c, int stage) {
    const int left = kend - c * KC;  // > 0
    char* const base = lds + stage * 2 * CHUNK;
    const __amdgpu_buffer_rsrc_t rK =
        make_rsrc(Kp + (int64_t)c * KC * a.ldk * 2, (uint32_t)(((left - 1) * a.ldk + a.d) * 2));
    const __amdgpu_buffer_rsrc_t rV =
        make_rsrc(Vp + (int64_t)c * KC * a.ldv * 2, (uint32_t)(((left - 1) * a.ldv + a.d) * 2));
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      load_lds16(rK, (HXMI_LDS void*)to_lds(base + (i * NW + w) * 1024), ko[i]);
      load_lds16(rV, (HXMI_LDS void*)to_lds(base + CHUNK + (i * NW + w) * 1024), vo[i]);
    }
  };

  float16v oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) oacc[t] = float16v{};
  float m_run = -INFINITY, l_run = 0.f;
  // This lane's K fragment of step st and V^T fragment of output tile dt in
  // a stage sit at kbase[st] / vbase[dt] plus a multiple of 32 / 4 rows:
  // neither swizzle changes over those.
  int kbase[DS], vbase[DT];
#pragma unroll
  for (int st = 0; st < DS; ++st) kbase[st] = k_off<D>(lane & 31, st * 2 + h);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int g = lane >> 4, L = lane & 15;
    const int d = dt * 32 + ((g & 1) << 4) + ((L & 3) << 2);
    vbase[dt] = CHUNK + v_off<D>(4 * h + (L >> 2), d >> 3) + (d & 7) * 2;
  }

  // Mask entries of the 32-key block at kb < skv, keys kb + 16h to + 16h + 15
  // of this lane's query as they lie in memory.  A lane's scores are keys
  // kb + 8g + 4h + j: the halves change places between the two lanes of a
  // query when they are used (8-byte loads in the scores' own order touch
  // every line of the mask twice as often).
  auto mask_vals = [&](int kb, MaskBlock& mk) {
    if (kb + 32 <= a.skv) {  // (wave-uniform)
#pragma unroll
      for (int x = 0; x < 2; ++x) mk.v[x] = *(const int4u*)(mrow + kb + 16 * h + 8 * x);
    } else {
      _Float16 e[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) e[i] = mrow[min(kb + 16 * h + i, a.skv - 1)];
      __builtin_memcpy(mk.v, e, 32);
    }
  };

  // The group of keys from kb on, its K rows at `rows` in LDS.  EDGE: some
  // of the keys may be past the sequence or the causal limit.
  auto group = [&](auto EDGE_, int kb, const char* rows, const MaskBlock (&mk)[MASK ? NB : 1]) {
    constexpr int N = NB;
    constexpr bool SCALED = decltype(EDGE_)::value;  // scores multiplied by a.c before the maximum
    // S: D[key][query], lane holds query lane%32, keys 8g + 4h + j of each
    // block.  Fragments are read one step ahead of their MFMAs; the
    // scheduling barriers keep the compiler from reading them all first,
    // which costs the registers of a wave per SIMD.
    float16v s[N];
    short8v kf[2][N], vf[2][DT];
    auto read_k = [&](int st) {
#pragma unroll
      for (int n = 0; n < N; ++n) kf[st & 1][n] = *(const short8v*)(rows + kbase[st] + n * 32 * RB);
    };
    // V^T of the 16-key step u: keys {16u + 4h + j, 16u + 8 + 4h + j}, at
    // rows 16 u (+ 8) past this lane's V base
    auto read_v = [&](int u) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const char* vb = rows + vbase[dt] + 16 * u * RB;
        const short4v lo = lds_read_tr16(vb);
        const short4v hi = lds_read_tr16(vb + 8 * RB);
        vf[u & 1][dt] = short8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    };
    read_k(0);
#pragma unroll
    for (int st = 0; st < DS; ++st) {
      if (st + 1 < DS) read_k(st + 1);
      else read_v(0);
#pragma unroll
      for (int n = 0; n < N; ++n) s[n] = Num<T>::mfma(kf[st & 1][n], qf[st], st == 0 ? float16v{} : s[n]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (SCALED) {
#pragma unroll
      for (int n = 0; n < N; ++n) {
        half4v me[4];  // by the g of the scores' keys
        if constexpr (MASK) {
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const int4v v = mk[n].v[x];
            const auto e0 = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
            const auto e1 = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
            me[x] = __builtin_bit_cast(half4v, uint2v{(uint32_t)e0[0], (uint32_t)e1[0]});
            me[2 + x] = __builtin_bit_cast(half4v, uint2v{(uint32_t)e0[1], (uint32_t)e1[1]});
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[n][i] *= a.c;
          if constexpr (MASK) s[n][i] = fmaf((float)me[i >> 2][i & 3], kLog2e, s[n][i]);
        }
      }
      if (kb + N * 32 > min(a.skv, q0 + a.causal_off + 1)) {  // (wave-uniform)
        const int last = min(a.skv - 1, qme + a.causal_off) - kb - 4 * h;
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (n * 32 + 8 * (i >> 2) + (i & 3) > last) s[n][i] = -INFINITY;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[n][i]);
    if constexpr (!SCALED) mx *= a.c;  // scale > 0
    mx = xor32_max(mx);
    const bool upd = mx > m_run + 8.0f;
    if (__any(upd)) {
      const float alpha = upd ? __builtin_amdgcn_exp2f(m_run - mx) : 1.0f;  // 0 on a first block
      if (upd) m_run = mx;
      l_run *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) oacc[t] *= alpha;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;  // every key so far masked: weights 0
    const float sc = SCALED ? 1.0f : a.c;
    // The weights of a step are taken while the MFMAs of the step before it
    // run.  The row sum uses the 16-bit weights P.V sees, so O is their
    // exact weighted average (a constant V comes back unchanged).
    float psum = 0.f;
    auto weights = [&](int u) {
      typename Num<T>::pair p2[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e = (u & 1) * 8 + 2 * i;
        p2[i] = typename Num<T>::pair{(T)__builtin_amdgcn_exp2f(fmaf(s[u >> 1][e], sc, -m_use)),
                                      (T)__builtin_amdgcn_exp2f(fmaf(s[u >> 1][e + 1], sc, -m_use))};
        psum = Num<T>::add_pair(p2[i], psum);
      }
      short8v pf;
      __builtin_memcpy(&pf, p2, 16);
      return pf;
    };
    short8v pf = weights(0);
#pragma unroll
    for (int u = 0; u < 2 * N; ++u) {
      short8v pn = pf;
      if (u + 1 < 2 * N) {
        read_v(u + 1);
        pn = weights(u + 1);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] = Num<T>::mfma(vf[u & 1][dt], pf, oacc[dt]);
      pf = pn;
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += psum;
  };

  // Two stages, one barrier a stage: past the barrier every wave's loads of
  // stage c have landed and every wave is done with stage c - 1, which
  // takes the loads of stage c + 1 while stage c is computed.  The first two
  // stages are issued together.  (One stage: its loads wait until every wave
  // is done with it, and only the other workgroup of the CU covers them.)
  auto stage_in = [&](int c) {
    if (ST == 1 && c > 0) {
      barrier_before_refill();
      issue(c, 0);
    }
    if (ST == 2 && c == 0 && nchunk > 1) wait_vmcnt<2 * LPW>();
    else wait_vmcnt0();
    barrier_before_refill();
  };
  auto stage_out = [&](int c) {
    if (ST == 2 && c > 0 && c + 1 < nchunk) issue(c + 1, (c + 1) & 1);
  };
  auto stage_at = [&](int c) { return lds + (c & (ST - 1)) * 2 * CHUNK; };
  // Leading stages that no wave needs the edge form for (a uniform count:
  // the waves meet at the barriers), then the rest.
  int nfull = 0;
  if constexpr (!MASK) nfull = max(0, min(a.skv, qb0 + a.causal_off + 1) / KC);
  // A stage's mask entries are loaded one stage ahead (before that stage's K
  // and V: loads return in order), so their latency passes under a stage's
  // MFMAs.
  MaskBlock mk[MASK ? GPC : 1][MASK ? NB : 1], mk_next[MASK ? GPC : 1][MASK ? NB : 1];
  auto load_mask = [&](int c, auto& m) {
    if constexpr (MASK) {
#pragma unroll
      for (int g = 0; g < GPC; ++g)
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          const int kb = c * KC + ((g * KS + kh) * NB + n) * 32;
          if (kb < wkend) mask_vals(kb, m[g][n]);
        }
    }
  };
  load_mask(0, mk);
  if (nchunk > 0) issue(0, 0);
  if (ST == 2 && nchunk > 1) issue(1, 1);
  int c = 0;
  for (; c < min(nfull, nchunk); ++c) {
    stage_in(c);
    stage_out(c);
#pragma unroll
    for (int g = 0; g < GPC; ++g) {
      const int row = (g * KS + kh) * NB * 32;
      group(std::false_type{}, c * KC + row, stage_at(c) + row * RB, mk[0]);
    }
  }
  for (; c < nchunk; ++c) {
    stage_in(c);
    load_mask(c + 1, mk_next);
    stage_out(c);
#pragma unroll
    for (int g = 0; g < GPC; ++g) {
      const int row = (g * KS + kh) * NB * 32;
      if (c * KC + row < wkend)
        group(std::true_type{}, c * KC + row, stage_at(c) + row * RB, mk[MASK ? g : 0]);
    }
    if constexpr (MASK) {
#pragma unroll
      for (int g = 0; g < GPC; ++g)
#pragma unroll
        for (int n = 0; n < NB; ++n) mk[g][n] = mk_next[g][n];
    }
  }

  // merge the key-split partials of each query group into wave kh = 0
  if constexpr (KS > 1) {
    constexpr int NV = Sh::NV;
    __syncthreads();  // every wave is done with the K / V chunk
    float* red = (float*)lds;
    if (kh > 0) {
      float* dst = red + ((kh - 1) * QG + qg) * NV * 64 + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) dst[(t * 16 + i) * 64] = oacc[t][i];
      dst[DT * 16 * 64] = m_run;
      dst[(DT * 16 + 1) * 64] = l_run;
    }
    __syncthreads();
    if (kh > 0) return;
#pragma unroll
    for (int o = 1; o < KS; ++o) {
      const float* src = red + ((o - 1) * QG + qg) * NV * 64 + lane;
      const float m2 = src[DT * 16 * 64], l2 = src[(DT * 16 + 1) * 64];
      const float mn = fmaxf(m_run, m2);
      const float a1 = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - mn);
      const float a2 = m2 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m2 - mn);
      l_run = l_run * a1 + l2 * a2;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[t][i] = oacc[t][i] * a1 + src[(t * 16 + i) * 64] * a2;
      m_run = mn;
    }
  }

  // O = D[d][query]: lane holds query lane%32, d = 32 dt + 8 g + 4 h + j
  const float l_tot = xor32_sum(l_run);
  const float inv = 1.0f / l_tot;
  if (qme < a.sq) {
    char* O = a.o + ((int64_t)bh * a.bo + (int64_t)qme * a.ldo) * 2;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (PART && dt * 32 + 8 * g + 4 * h >= a.d) continue;
        T o4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o4[j] = (T)(oacc[dt][4 * g + j] * inv);
        *(short4v*)(O + (dt * 32 + 8 * g + 4 * h) * 2) = __builtin_bit_cast(short4v, o4);
      }
  }
}

template <typename T, int D, int DT, bool PART, int QG, int KS, bool DEEP = false>
hipError_t launch_cfg(AArgs a, const AttnProblem& p, bool mask, hipStream_t stream) {
  if constexpr (!AttnShape<D, QG, KS, false, DEEP>::ok) {
    return hipErrorNotSupported;
  } else {
    a.nqb = (int)((p.s + 32 * QG - 1) / (32 * QG));
    const int64_t blocks = p.bh * a.nqb;
    if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
    a.order = !p.causal ? ORDER_SLICES : (blocks <= 512 ? ORDER_PAIRED : ORDER_HEAVY);
    const dim3 grid((unsigned)blocks), block(64 * QG * KS);
    if (mask)
      hipLaunchKernelGGL((attention_fwd<T, D, DT, PART, QG, KS, true, DEEP>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((attention_fwd<T, D, DT, PART, QG, KS, false, DEEP>), grid, block, 0, stream, a);
    return hipGetLastError();
  }
}

// The head-dim rows (D, DT, PART) of p at workgroup shape cfg; shapes that
// only the tuning knob asks for exist for fp16 head dims 64 and 128.
template <typename T, int D, int DT, bool PART>
hipError_t launch_d(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream) {
  const bool m = p.mask != nullptr;
  switch (cfg) {
    case 41: return launch_cfg<T, D, DT, PART, 4, 1>(a, p, m, stream);
    case 14:
      // One workgroup a CU at most: its loads need a second stage to pass
      // under its MFMAs (2 x 1968 x 1968 causal, D 128: 22.9 -> 20.9 us, 16 x
      // 458 10.5 -> 9.8); from 257 workgroups on two share a CU, which only
      // one stage each allows (8 x 1132: 20.0 us, two stages 27.6).
      if (D > 64 && p.bh * ((p.s + 31) / 32) <= 256) return launch_cfg<T, D, DT, PART, 1, 4, (D > 64)>(a, p, m, stream);
      return launch_cfg<T, D, DT, PART, 1, 4>(a, p, m, stream);
    case 42: return launch_cfg<T, D, DT, PART, 4, 2>(a, p, m, stream);
    case 22: return launch_cfg<T, D, DT, PART, 2, 2>(a, p, m, stream);
    default: break;
  }
  if constexpr (std::is_same_v<T, _Float16> && !PART) {
    switch (cfg) {
      case 21: return launch_cfg<T, D, DT, PART, 2, 1>(a, p, m, stream);
      case 12: return launch_cfg<T, D, DT, PART, 1, 2>(a, p, m, stream);
      case 24: return launch_cfg<T, D, DT, PART, 2, 4>(a, p, m, stream);
      default: break;
    }
  }
  return hipErrorNotSupported;
}

template <typename T>
hipError_t launch_t(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream) {
  if (p.d == 64) return launch_d<T, 64, 2, false>(a, p, cfg, stream);
  if (p.d == 128) return launch_d<T, 128, 4, false>(a, p, cfg, stream);
  if (p.d < 64) return launch_d<T, 64, 2, true>(a, p, cfg, stream);
  return p.d <= 96 ? launch_d<T, 128, 3, true>(a, p, cfg, stream) : launch_d<T, 128, 4, true>(a, p, cfg, stream);
}

}  // namespace attn
}  // namespace hxmi
