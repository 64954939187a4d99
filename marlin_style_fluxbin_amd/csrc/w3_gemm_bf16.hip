// Instantiations of the W3 GEMM: bf16 activations, up to 48 activation rows per workgroup.
#include "w3_gemm.h"

namespace fx {
bool dispatch_gemm_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s) {
  if (p.nk != 8) return false;
  switch (p.rt * 10 + p.mt) {
    case 11: return gemm_launch<kBF16, 1, 1, 8, 3, false>(p, a, s);
    case 21: return gemm_launch<kBF16, 2, 1, 8, 3, false>(p, a, s);
    case 31: return gemm_launch<kBF16, 3, 1, 8, 3, false>(p, a, s);
    case 12: return gemm_launch<kBF16, 1, 2, 8, 1, false>(p, a, s);
    case 22: return gemm_launch<kBF16, 2, 2, 8, 1, false>(p, a, s);
    case 32: return gemm_launch<kBF16, 3, 2, 8, 1, false>(p, a, s);
    case 13: return gemm_launch<kBF16, 1, 3, 8, 1, false>(p, a, s);
    case 23: return gemm_launch<kBF16, 2, 3, 8, 1, false>(p, a, s);
    case 33: return gemm_launch<kBF16, 3, 3, 8, 1, false>(p, a, s);
  }
  return false;
}
}  // namespace fx
