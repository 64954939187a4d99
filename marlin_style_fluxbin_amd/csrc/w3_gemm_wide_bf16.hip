// Instantiations of the W3 GEMM: bf16 activations, 64 to 128 activation rows per workgroup.
#include "w3_gemm.h"

namespace fx {
bool dispatch_gemm_wide_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s) {
  if (p.nk == 8 && p.mt == 4 && p.rt == 2) return gemm_launch<kBF16, 2, 4, 8, 1, false>(p, a, s);
  if (p.nk == 8 && p.mt == 4 && p.rt == 3) return gemm_launch<kBF16, 3, 4, 8, 1, false>(p, a, s);
  if (p.nk == 8 && p.mt == 7 && p.rt == 2) return gemm_launch<kBF16, 2, 7, 8, 1, false>(p, a, s);
  if (p.nk == 4 && p.mt == 7 && p.rt == 4) return gemm_launch<kBF16, 4, 7, 4, 1, true>(p, a, s);
  if (p.nk == 4 && p.mt == 8 && p.rt == 2) return gemm_launch<kBF16, 2, 8, 4, 1, true>(p, a, s);
  if (p.nk == 4 && p.mt == 8 && p.rt == 4) return gemm_launch<kBF16, 4, 8, 4, 1, true>(p, a, s);
  return false;
}
}  // namespace fx
