// Dense [O, K] weight of a hybrid g128/s8 two-base layout (deployment.py:118-121 ->
// evaluation.py:59-175), the dequantize of PackedHybridLinear's dense fallback.
//
// Every value is formed in fp32 in the reference's order (per base (sign * row) *
// column added to a zero start, the refinement formed the same way and added at
// its column) and rounded once, so the weight is bitwise that of the torch
// arithmetic; contraction to fused multiply-adds would move its last bit.
//
// Bound by the store of 2 O K bytes.  A workgroup owns 128 columns (one group) of
// kHyRestoreRows rows: lane c of a row's 16 lanes expands byte c of the two sign
// rows into 8 columns and stores them as 16 bytes, so a row's 256 bytes leave
// together; the group's column scales and the refinement column of each of the
// lane's 8 columns stay in registers over the rows.  Layout data that the torch
// arithmetic refuses (a scale that is not finite, refinement columns outside the
// group or not ascending) sets *bad; such columns are not written through.
//
// Measured: the fallback of a Qwen3-8B layer's seven Linears on 200 rows took
// 13.8 ms with the torch arithmetic (about thirty passes over fp32 and int8
// [O, K] tensors and four host synchronisations each) and takes 0.52 ms with this
// kernel and one wait.
#include "common.h"
#include "two_base_launch.h"

#pragma clang fp contract(off)

namespace fx {

constexpr int kHyRestoreRows = 128;  // rows per workgroup, 16 at a time

// The even bits of a 16-bit value, packed (interleaved two-base codes: base b of
// column i at bit 2 i + b).
__device__ __forceinline__ unsigned even_bits(unsigned v) {
  v &= 0x5555u;
  v = (v | (v >> 1)) & 0x3333u;
  v = (v | (v >> 2)) & 0x0f0fu;
  return (v | (v >> 4)) & 0xffu;
}
__device__ __forceinline__ float signed_scale(unsigned bit, float v) {  // bit ? v : -v
  return __uint_as_float(__float_as_uint(v) ^ ((bit ^ 1u) << 31));
}
__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }

template <int WDT>
__global__ __launch_bounds__(256) void hybrid_restore_kernel(HybridRestoreArgs a) {
  const int c = int(threadIdx.x & 15u), r0 = int(threadIdx.x >> 4);
  const int g = int(blockIdx.x % unsigned(a.G));
  const int o0 = int(blockIdx.x / unsigned(a.G)) * kHyRestoreRows;
  bool bad = false;
  float col[8][2], ucol[8][2];
  unsigned slot = 0;  // a nibble per column: refinement slot + 1, or 0
  {
    const float* cols = a.columns + (size_t(g) * 128 + c * 8) * 2;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        col[e][b] = cols[2 * e + b];
        ucol[e][b] = 0.f;
        bad |= not_finite(col[e][b]);
      }
    }
    int previous = -1;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int idx = a.indices[size_t(g) * 8 + s];
      const float s0 = a.sparse_columns[(size_t(g) * 8 + s) * 2], s1 = a.sparse_columns[(size_t(g) * 8 + s) * 2 + 1];
      bad |= idx <= previous || idx > 127 || not_finite(s0) || not_finite(s1);
      previous = idx;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (idx == c * 8 + e) {
          ucol[e][0] = s0;
          ucol[e][1] = s1;
          slot |= unsigned(s + 1) << (4 * e);
        }
      }
    }
  }
#pragma unroll 2
  for (int i = r0; i < kHyRestoreRows; i += 16) {
    const int o = o0 + i;
    if (o >= a.O) break;
    const size_t go = size_t(g) * a.O + o;
    unsigned p0, p1, q0, q1;
    if (a.interleaved) {
      const unsigned pair = *reinterpret_cast<const uint16_t*>(a.codes + go * 32 + 2 * c);
      const unsigned spair = *reinterpret_cast<const uint16_t*>(a.sparse_codes + go * 2);
      p0 = even_bits(pair), p1 = even_bits(pair >> 1);
      q0 = even_bits(spair), q1 = even_bits(spair >> 1);
    } else {
      p0 = a.codes[go * 32 + c], p1 = a.codes[go * 32 + 16 + c];
      q0 = a.sparse_codes[go * 2], q1 = a.sparse_codes[go * 2 + 1];
    }
    const float2 row = *reinterpret_cast<const float2*>(a.rows + go * 2);
    const float2 srow = *reinterpret_cast<const float2*>(a.sparse_rows + go * 2);
    bad |= not_finite(row.x) || not_finite(row.y) || not_finite(srow.x) || not_finite(srow.y);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t0 = signed_scale((p0 >> e) & 1u, row.x) * col[e][0];
      const float t1 = signed_scale((p1 >> e) & 1u, row.y) * col[e][1];
      v[e] = (0.f + t0) + t1;
    }
    if (slot) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned s = (slot >> (4 * e)) & 15u;
        if (s) {
          const float u0 = signed_scale((q0 >> (s - 1)) & 1u, srow.x) * ucol[e][0];
          const float u1 = signed_scale((q1 >> (s - 1)) & 1u, srow.y) * ucol[e][1];
          v[e] = v[e] + ((0.f + u0) + u1);
        }
      }
    }
    const size_t at = size_t(o) * (size_t(a.G) * 128) + size_t(g) * 128 + c * 8;
    if constexpr (WDT == kF32) {
      float4* dst = reinterpret_cast<float4*>(static_cast<float*>(a.weight) + at);
      dst[0] = make_float4(v[0], v[1], v[2], v[3]);
      dst[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      uint4 w;
      unsigned* pair = reinterpret_cast<unsigned*>(&w);
#pragma unroll
      for (int e = 0; e < 8; e += 2)
        pair[e >> 1] = unsigned(from_f32<WDT>(v[e])) | (unsigned(from_f32<WDT>(v[e + 1])) << 16);
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.weight) + at) = w;
    }
  }
  if (bad) *a.bad = 1;  // every writer stores the same value
}

void launch_hybrid_restore(int weight_dtype, const HybridRestoreArgs& a, hipStream_t stream) {
  const dim3 grid(unsigned((a.O + kHyRestoreRows - 1) / kHyRestoreRows) * unsigned(a.G)), block(256);
  if (weight_dtype == kF32)
    hipLaunchKernelGGL(hybrid_restore_kernel<kF32>, grid, block, 0, stream, a);
  else if (weight_dtype == kBF16)
    hipLaunchKernelGGL(hybrid_restore_kernel<kBF16>, grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL(hybrid_restore_kernel<kF16>, grid, block, 0, stream, a);
}

}  // namespace fx
