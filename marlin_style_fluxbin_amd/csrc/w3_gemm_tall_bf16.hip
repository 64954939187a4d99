// Instantiation of the W3 GEMM for many activation rows: bf16 activations.
#include "w3_gemm_tall.h"

namespace fx {
bool dispatch_gemm_tall_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s) {
  return p.mt == kTallRowTiles && gemm_tall_launch<kBF16, kTallRowTiles, kTallWaves>(p, a, s);
}
}  // namespace fx
