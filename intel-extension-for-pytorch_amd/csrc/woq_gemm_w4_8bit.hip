// The prefill kernel's launches of 8-bit weights, fp16 or bf16 compute: twice the tile bytes per K step.
#include "woq_gemm_w4.h"

namespace woq {

// 8-bit weights of one shape: integers or float8 bytes, fp16 or bf16 compute
template <class S>
static int launch8(const FpArgs& f, int regime, int g_shift, hipStream_t st, int splits, const SplitKScratch* scratch) {
  if (f.fp8)
    return regime == kRegimeF16 ? launch_shape<kRegimeF16, S, 8, true>(f, g_shift, st, splits, scratch)
                                : launch_shape<kRegimeBF16, S, 8, true>(f, g_shift, st, splits, scratch);
  return regime == kRegimeF16 ? launch_shape<kRegimeF16, S, 8>(f, g_shift, st, splits, scratch)
                              : launch_shape<kRegimeBF16, S, 8>(f, g_shift, st, splits, scratch);
}

int launch_gemm_w4_8bit(const FpArgs& f, int regime, int g_shift, hipStream_t st, int shape, int splits, const SplitKScratch* scratch) {
  return shape == 42  ? launch8<G4Shape<4, 2>>(f, regime, g_shift, st, splits, scratch)
         : shape == 5 ? launch8<G4Shape<8, 2, 8>>(f, regime, g_shift, st, splits, scratch)
                      : launch8<G4Shape<8, 2>>(f, regime, g_shift, st, splits, scratch);
}

}  // namespace woq
