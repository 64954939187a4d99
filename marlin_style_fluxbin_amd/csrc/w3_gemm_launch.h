// Host-side declarations of the W3 GEMM (w3_gemm.h, w3_gemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fx {

constexpr int kGemmMaxRows = 8192;  // activation rows per call (64 row blocks and more)

struct GemmArgs {
  const uint4* packed;  // gemm_pack_kernel's: [ceil(M / 16 MT)][batch][step 16][MT][lane 64]
  const uint8_t* planes;
  const uint16_t* scales;
  const uint8_t* zeros;  // null: zero-point 4
  const uint16_t* bias;  // [O] in x's type, or null
  float* partial;        // null: write out directly (one K split)
  uint16_t* out;         // [M, O]
  int M, O, G;
  int sdt;                // scale dtype
  int batches_per_split;  // four-group batches of a K split (grid z)
  int vec;                // O a multiple of 4 and out / partial aligned to 4 elements
};

struct GemmPackArgs {
  const uint16_t* x;    // [M, K], 16-byte aligned
  const int16_t* perm;  // [K] (16-byte aligned) or null: the identity
  uint4* packed;
  int M, K, mt;         // mt: 16-row tiles per row block
};

// A tiling: rt 16-row output tiles x mt 16-row activation tiles per workgroup, nk
// waves dealing its K range.
struct GemmPlan {
  int rt, mt, nk;
  int splits, batches_per_split;
  bool tall;  // w3_gemm_tall.h: kTallTiles kTallWaves output tiles x kTallRowTiles
};
constexpr int kTallTiles = 3, kTallWaves = 4, kTallRowTiles = 8;

// Instantiated (rt, mt, nk): (1..3, 1..3, 8) (2..3, 4, 8) (2, 7, 8) (4, 7, 4) (2, 8, 4)
// (4, 8, 4).  False otherwise.
bool dispatch_gemm_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
bool dispatch_gemm_f16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
bool dispatch_gemm_wide_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
bool dispatch_gemm_wide_f16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
bool dispatch_gemm_tall_bf16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
bool dispatch_gemm_tall_f16(const GemmPlan& p, const GemmArgs& a, hipStream_t s);
void launch_gemm_pack(const GemmPackArgs& a, hipStream_t s);
void launch_gemm_finish(int xdt, const GemmArgs& a, int splits, hipStream_t s);

}  // namespace fx
