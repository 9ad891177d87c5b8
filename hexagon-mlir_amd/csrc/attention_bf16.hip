// Instantiations of the fused attention for bf16 operands.
#include "attention_impl.h"

namespace hxmi {
namespace attn {

hipError_t launch_bf16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream) {
  return launch_t<__bf16>(a, p, cfg, stream);
}

}  // namespace attn
}  // namespace hxmi
