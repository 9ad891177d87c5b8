// Fused attention dispatch: the workgroup shape and the launch arguments.
#include "attention_impl.h"

namespace hxmi {
namespace attn {
hipError_t launch_f16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream);
hipError_t launch_bf16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream);
}  // namespace attn

namespace {

// Launch shape: query waves x key-split waves per workgroup.
int pick_cfg(const AttnProblem& p) {
  const int64_t forced = knob(KNOB_ATTN_CFG);
  if (forced != KNOB_UNSET) return (int)forced;
  // Enough 128-query workgroups to cover most CUs: 4 query waves (x2 key
  // splits at D = 64, where the merge fits in LDS); otherwise one query group
  // per workgroup with the keys split over 4 waves (ViT-B/16 batch 8: 7.3 us
  // against 7.6 / 10.8; a 32-head 512-token causal prefill: 8.3 us against
  // 10.9 / 11.3, measured on MI355X)
  const int64_t wg4 = p.bh * ((p.s + 127) / 128);
  if (wg4 >= 192) return p.d <= 64 ? 42 : 41;
  return 14;
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
  a.mask_vec = p.mask && p.ldm % 4 == 0 && p.sm % 4 == 0 && ((uintptr_t)p.mask & 7) == 0;
  a.kbytes = (uint32_t)(((p.skv - 1) * p.ldk + p.d) * 2);
  a.vbytes = (uint32_t)(((p.skv - 1) * p.ldv + p.d) * 2);
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
  const int cfg = pick_cfg(p);
  return p.dtype == DT_BF16 ? attn::launch_bf16(a, p, cfg, stream) : attn::launch_f16(a, p, cfg, stream);
}

}  // namespace hxmi
