// Instantiations of the MFMA GEMM for operand rows off the 16-byte grid (fp16
// / bf16): contiguous matrices with an odd number of columns, views at odd
// element offsets.  Two tiles, as for ragged K: 128x128 (4 waves) for
// problems with enough of them to cover the CUs, 64x64 otherwise.
#include "gemm_impl.h"

namespace hxmi {
namespace gemm {
namespace {

template <bool NN, typename T, int EPI, bool OUTF32, bool RMS = false>
hipError_t any_tile(int tile, const KArgs& k, hipStream_t s) {
  if (tile == TILE_128x128) return launch_one<TILE_128x128, NN, T, EPI, OUTF32, false, RMS, false, true>(k, s);
  return launch_one<TILE_64x64, NN, T, EPI, OUTF32, false, RMS, false, true>(k, s);
}

template <typename T>
hipError_t any_t(int tile, bool nn, int epi, bool rms, const KArgs& k, hipStream_t s) {
  if (nn) return epi == EPI_BIAS ? any_tile<true, T, EPI_BIAS, false>(tile, k, s)
                                 : any_tile<true, T, EPI_NONE, false>(tile, k, s);
  switch (epi) {
    case EPI_BIAS: return rms ? any_tile<false, T, EPI_BIAS, false, true>(tile, k, s)
                              : any_tile<false, T, EPI_BIAS, false>(tile, k, s);
    case EPI_SILU_MUL: return rms ? any_tile<false, T, EPI_SILU_MUL, false, true>(tile, k, s)
                                  : any_tile<false, T, EPI_SILU_MUL, false>(tile, k, s);
    case EPI_GELU_TANH: return any_tile<false, T, EPI_GELU_TANH, false>(tile, k, s);
    case EPI_BIAS_GELU_TANH: return any_tile<false, T, EPI_BIAS_GELU_TANH, false>(tile, k, s);
    default: return rms ? any_tile<false, T, EPI_NONE, false, true>(tile, k, s)
                        : any_tile<false, T, EPI_NONE, false>(tile, k, s);
  }
}

}  // namespace

// (the combinations any_alignment_ok admits)
hipError_t launch_fast_unaligned(int tile, bool bf16, bool nn, int epi, bool out_f32, bool rms, const KArgs& k,
                                 hipStream_t s) {
  if (out_f32) return nn ? any_tile<true, _Float16, EPI_NONE, true>(tile, k, s)
                         : any_tile<false, _Float16, EPI_NONE, true>(tile, k, s);
  return bf16 ? any_t<__bf16>(tile, nn, epi, rms, k, s) : any_t<_Float16>(tile, nn, epi, rms, k, s);
}

}  // namespace gemm
}  // namespace hxmi
