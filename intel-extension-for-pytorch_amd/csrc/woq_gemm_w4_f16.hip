// The prefill kernel's launches of 4-bit weights under fp16 compute.
#include "woq_gemm_w4.h"

namespace woq {

int launch_gemm_w4_f16(const FpArgs& f, int g_shift, hipStream_t st, int shape, int splits, const SplitKScratch* scratch) {
  return launch_w4_4bit<kRegimeF16>(f, g_shift, st, shape, splits, scratch);
}

}  // namespace woq
