// Dense [O, K] weight of a hybrid g128/s8 two-base layout (deployment.py:118-121 ->
// evaluation.py:59-175), the dequantize of PackedHybridLinear's dense fallback.
//
// Every value is formed in fp32 in the reference's order (per base (sign * row) *
// column added to a zero start, the refinement formed the same way and added at
// its column) and rounded once, so the weight is bitwise that of the torch
// arithmetic; contraction to fused multiply-adds would move its last bit.
//
// Bound by the store of 2 O K bytes.  A workgroup owns 128 columns (one group) of
// kHyRestoreRows rows, a wave eight rows at a time: lane c of a row's 16 lanes expands
// byte c of the two sign rows into 8 columns, with the group's column scales kept in
// registers over the rows, and leaves them in the wave's LDS rows; then each of the 64
// lanes forms one refined column (8 rows x 8 columns, their scales in registers too)
// and writes it over, and the rows leave as 16-byte stores, 256 bytes of a row
// together.  (Selecting the refined columns within each lane's eight instead cost more
// than the rest of the kernel: they are one in sixteen.)  Layout data that the torch
// arithmetic refuses (a scale that is not finite, refinement columns outside the
// group or not ascending) sets *bad; such columns are not written through.
//
// Measured: the fallback of a Qwen3-8B layer's seven Linears on 200 rows took
// 13.8 ms with the torch arithmetic (about thirty passes over fp32 and int8
// [O, K] tensors and four host synchronisations each) and takes 0.47 ms with this
// kernel and one wait, bound by the host (this kernel 148 us of it, the products 162; a
// check launch of its own, so that the host waits less, gained nothing).  The seven
// launches' mean is 21.3 us (32.5 with the refined columns selected in registers).
#include "common.h"
#include "two_base_launch.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace fx {

constexpr int kHyRestoreTurns = 2;                     // eight-row turns of a wave, all loaded ahead
constexpr int kHyRestoreRows = 32 * kHyRestoreTurns;  // rows per workgroup

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

// One weight: (0 + row0 column0) + row1 column1 with the signs' bits (1 = +).
__device__ __forceinline__ float two_base(unsigned s0, unsigned s1, const float2& row, float c0, float c1) {
  return (0.f + signed_scale(s0, row.x) * c0) + signed_scale(s1, row.y) * c1;
}

template <int WDT>
__global__ __launch_bounds__(256) void hybrid_restore_kernel(HybridRestoreArgs a) {
  using Element = std::conditional_t<WDT == kF32, float, uint16_t>;
  typedef Element __attribute__((may_alias)) StagedElement;  // one value of a staged vector
  constexpr int kVecs = 8 * int(sizeof(Element)) / 16;  // 16-byte vectors of 8 columns
  __shared__ u32x4_t stage[4][8][16 * kVecs];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int c = lane & 15;
  const int g = int(blockIdx.x % unsigned(a.G));
  const int o0 = int(blockIdx.x / unsigned(a.G)) * kHyRestoreRows;
  bool bad = false;
  float col[8][2];
  {
    const float* cols = a.columns + (size_t(g) * 128 + c * 8) * 2;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        col[e][b] = cols[2 * e + b];
        bad |= not_finite(col[e][b]);
      }
    }
  }
  // the lane's refined column: slot lane % 8, of rows lane / 8
  const int slot = lane & 7;
  const int16_t* indices = a.indices + size_t(g) * 8;
  const int index = indices[slot];
  bad |= index < 0 || index > 127 || (slot > 0 && index <= indices[slot > 0 ? slot - 1 : 0]);
  const int at = index & 127;  // inside the group; a bad index is reported
  const float2 ucol = *reinterpret_cast<const float2*>(a.sparse_columns + (size_t(g) * 8 + slot) * 2);
  const float2 rcol = *reinterpret_cast<const float2*>(a.columns + (size_t(g) * 128 + at) * 2);
  bad |= not_finite(ucol.x) || not_finite(ucol.y);
  // raw sign bytes of one row: an interleaved pair, or the two planes' bytes
  const auto signs = [&](const uint8_t* codes, int byte, int width) -> unsigned {
    if (a.interleaved) return *reinterpret_cast<const uint16_t*>(codes + 2 * byte);
    return unsigned(codes[byte]) | (unsigned(codes[width + byte]) << 8);
  };
  const auto base0 = [&](unsigned v) { return a.interleaved ? even_bits(v) : v & 0xffu; };
  const auto base1 = [&](unsigned v) { return a.interleaved ? even_bits(v >> 1) : v >> 8; };
  struct Turn {
    unsigned codes[2], patch, sparse;  // of the lane's two rows; of its refined column's row
    float2 row[2], prow, srow;
  } turn[kHyRestoreTurns];
#pragma unroll
  for (int k = 0; k < kHyRestoreTurns; ++k) {  // rows past O read the last row and are not stored
    const int i = o0 + wave * 8 * kHyRestoreTurns + 8 * k;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const size_t go = size_t(g) * a.O + min(i + 4 * h + (lane >> 4), a.O - 1);
      turn[k].codes[h] = signs(a.codes + go * 32, c, 16);
      turn[k].row[h] = *reinterpret_cast<const float2*>(a.rows + go * 2);
    }
    const size_t go = size_t(g) * a.O + min(i + (lane >> 3), a.O - 1);
    turn[k].patch = signs(a.codes + go * 32, at >> 3, 16);
    turn[k].sparse = signs(a.sparse_codes + go * 2, 0, 1);
    turn[k].prow = *reinterpret_cast<const float2*>(a.rows + go * 2);
    turn[k].srow = *reinterpret_cast<const float2*>(a.sparse_rows + go * 2);
  }
#pragma unroll
  for (int k = 0; k < kHyRestoreTurns; ++k) {
    const Turn& in = turn[k];
    const int i = o0 + wave * 8 * kHyRestoreTurns + 8 * k;
    if (i >= a.O) break;  // wave-uniform
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned p0 = base0(in.codes[h]), p1 = base1(in.codes[h]);
      bad |= not_finite(in.row[h].x) || not_finite(in.row[h].y);
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = two_base((p0 >> e) & 1u, (p1 >> e) & 1u, in.row[h], col[e][0], col[e][1]);
      u32x4_t* dst = &stage[wave][4 * h + (lane >> 4)][c * kVecs];
      if constexpr (WDT == kF32) {
        dst[0] = u32x4_t{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
        dst[1] = u32x4_t{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])};
      } else {
        unsigned pair[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) pair[e] = round_pair_bits<WDT>(v[2 * e], v[2 * e + 1]);
        dst[0] = u32x4_t{pair[0], pair[1], pair[2], pair[3]};
      }
    }
    {
      const unsigned p0 = base0(in.patch), p1 = base1(in.patch), q0 = base0(in.sparse), q1 = base1(in.sparse);
      bad |= not_finite(in.srow.x) || not_finite(in.srow.y);
      const float w = two_base((p0 >> (at & 7)) & 1u, (p1 >> (at & 7)) & 1u, in.prow, rcol.x, rcol.y) +
                      two_base((q0 >> slot) & 1u, (q1 >> slot) & 1u, in.srow, ucol.x, ucol.y);
      wave_lds_order();  // after the row's own values
      StagedElement* dst = reinterpret_cast<StagedElement*>(&stage[wave][lane >> 3][0]) + at;
      if constexpr (WDT == kF32) *dst = w;
      else *dst = from_f32<WDT>(w);
      wave_lds_order();
    }
#pragma unroll
    for (int n = 0; n < 2 * kVecs; ++n) {
      const int unit = n * 64 + lane, rr = unit / (16 * kVecs), at16 = unit % (16 * kVecs);
      const u32x4_t v = stage[wave][rr][at16];
      const int o = i + rr;
      if (o < a.O)
        *reinterpret_cast<u32x4_t*>(static_cast<Element*>(a.weight) + size_t(o) * (size_t(a.G) * 128) + size_t(g) * 128 +
                                  at16 * (16 / int(sizeof(Element)))) = v;
    }
    wave_lds_order();
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
