// Instantiations of the fused attention for f16 operands.
#include "attention_impl.h"

namespace hxmi {
namespace attn {

hipError_t launch_f16(const AArgs& a, const AttnProblem& p, int cfg, hipStream_t stream) {
  return launch_t<_Float16>(a, p, cfg, stream);
}

}  // namespace attn
}  // namespace hxmi
