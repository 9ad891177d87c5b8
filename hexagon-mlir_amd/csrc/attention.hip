// Fused attention dispatch: the workgroup shape and the launch arguments.
#include <algorithm>

#include "attention_impl.h"

namespace hxmi {
namespace attn {
hipError_t launch_f16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream);
hipError_t launch_bf16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream);
}  // namespace attn

namespace {

// Launch shape: query waves x key-split waves per workgroup.
int pick_cfg(const AttnProblem& p) {
  // Queries per workgroup: the most that still spread over the chip, since
  // each workgroup reads its K and V through LDS once; 128 queries are split
  // over two halves of the keys to have eight waves (four with few keys, and
  // at head dims over 64, whose merge and registers allow no more).  us, graph replays on MI355X, 128 / 64 / 32
  // queries a workgroup:
  //   head dim 64, full:    96 x 197 keys (192 / 384 / 672 workgroups) 7.0 (8 waves: 7.3) / 7.5 / 9.9; 48 x 257
  //                         (144 / 240 / 432) 8.3 / 6.5 / 7.2; 32 x 577 (160 / 320 / 608) 10.7 / 11.5 /
  //                         13.6; 32 x 300 (96 / 160 / 320) 8.1 / 6.5 / 7.2; 8 x 2048 (128 / 256 / 512)
  //                         20.4 / 16.0 / 17.7; 4 x 2048 (64 / 128 / 256) 20.3 / 15.9 / 13.4
  //   head dim 64, causal:  32 x 2048 (512 / 1024 / 2048) 25.1 / 28.8 / 38.7; 32 x 1024 (256 / 512 /
  //                         1024) 13.8 / 11.3 / 15.4; 32 x 512 (128 / 256 / 512) 9.5 / 7.3 / 6.9
  // With few keys a key split over four waves costs more than it spreads,
  // once its workgroups no longer have a CU each (unmasked 48 x 157, 240 of
  // them 5.5, 64 queries 5.9; 48 x 177, 288: 6.7 and 5.9); and a causal
  // workgroup count of two per CU lets heavy and light blocks pair up, so the
  // causal lines lie at about twice the others.  Up to 224 keys a causal block
  // has one or two stages whatever its weight, and 128 queries pay from 192
  // workgroups on (96 x 197 6.5, 64 queries 7.0; head dim 128, 96 x 157 7.6
  // and 8.2, 192 x 100 7.3 and 8.1; but 96 x 256 10.1 and 9.5), masked calls
  // and the three-quarter rows of head dims 72-96 aside (96 x 197 masked 9.0
  // and 8.4, head dim 80 8.3 and 7.3).
  const bool few_keys = p.skv <= 384;
  const int64_t wg128 = p.bh * ((p.s + 127) / 128), wg64 = p.bh * ((p.s + 63) / 64),
                wg32 = p.bh * ((p.s + 31) / 32);
  // A mask's entries take registers that eight waves do not have: 128
  // queries run four waves, and pay only from 320 on (8 waves / 4 waves / 64
  // queries: 32 x 1024 full 23.7 / 25.5 / 20.8, 64 x 500 15.3 / 15.7 / 14.1,
  // 64 x 1000 39.1 / 38.7 / 40.3, 128 x 2048 causal 135 / 131 / 142).
  const bool masked64 = p.mask && p.d <= 64;
  const bool short_causal = p.causal && p.skv <= 224 && !p.mask && (p.d <= 64 || p.d > 96);
  if (wg128 >= (short_causal ? 192 : p.causal ? 320 : few_keys ? 192 : masked64 ? 320 : 144))
    return p.d <= 64 && !few_keys && !p.mask ? 42 : 41;
  // (64-192 keys at head dims over 64: the merge of four key splits takes as
  // long as the keys; 4 x 157 causal 6.4 us against 7.2, 32 x 155 full 7.4
  // against 7.5, 64 x 201 8.3 against 7.6)
  if (p.d > 64 && p.skv <= 192) return 22;
  if (few_keys) return wg64 >= 144 && (p.mask || wg32 > 256) ? 22 : 14;
  return wg64 >= (p.causal ? 288 : 192) ? 22 : 14;
}

}  // namespace

hipError_t launch_attention(const AttnProblem& p, hipStream_t stream) {
  if (p.bh == 0 || p.s == 0) return hipSuccess;
  attn::AArgs a{};
  a.q = (const char*)p.q;
  a.k = (const char*)p.k;
  a.v = (const char*)p.v;
  a.o = (char*)p.o;
  a.mask = (const char*)p.mask;
  a.bh = (int)p.bh;
  a.sq = (int)p.s;
  a.skv = (int)p.skv;
  a.d = (int)p.d;
  a.kv_group = (int)p.kv_group;
  a.mask_group = (int)(p.mask_group > 0 ? p.mask_group : 1);
  a.causal_off = p.causal == 1 ? 0 : p.causal == 2 ? (int)(p.skv - p.s) : (int)p.skv;
  a.ldq = p.ldq;
  a.ldk = p.ldk;
  a.ldv = p.ldv;
  a.ldo = p.ldo;
  a.ldm = p.ldm;
  a.bq = p.sq;
  a.bk = p.sk;
  a.bv = p.sv;
  a.bo = p.so;
  a.bm = p.sm;
  a.c = p.scale * attn::kLog2e;
  if (p.d % 8 || p.d < 8 || p.d > 128) return hipErrorNotSupported;
  const auto launch = [&](int cfg) {
    return p.dtype == DT_BF16 ? attn::launch_bf16(a, p, cfg, stream) : attn::launch_f16(a, p, cfg, stream);
  };
  // an override that has no instantiation for this type and head dim gives
  // way to the picked shape (nothing has been launched then)
  const int64_t forced = knob(KNOB_ATTN_CFG);
  const hipError_t e = forced == KNOB_UNSET ? hipErrorNotSupported : launch((int)std::clamp<int64_t>(forced, 0, 999));
  return e == hipErrorNotSupported ? launch(pick_cfg(p)) : e;
}

}  // namespace hxmi
