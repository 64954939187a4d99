// Exact weight values of a W3 g128 planar payload in registers, without arithmetic per
// weight: shared by the kernels that need round_x(round_scale(s (q - z))).
//
// A (row, group) has eight possible values.  A lane forms them once, rounded, and keeps
// their low and high bytes in two register pairs; v_perm_b32 is then an eight-entry
// byte lookup with four codes a register.
#pragma once
#include "common.h"

namespace fx {

// T_s from three-input bit operations (v_bitop3_b32, gfx950): u = M1 ? b : ~c
// (table 0xB1, operand order b, c, m: the inversion of stored plane 2 folded in),
// then T = M0 ? a : u (table 0xE4).  The complement of the shifted plane differs
// from the shifted complement only in shifted-in bits, which land in bits the
// masks take from the other planes or in the don't-care bit.  Two instructions
// per T_s where the compiler's own rewrite of the inserts took three to four.
__device__ __forceinline__ unsigned select3(unsigned a, unsigned b, unsigned c, unsigned m0, unsigned m1) {
  return __builtin_amdgcn_bitop3_b32(a, __builtin_amdgcn_bitop3_b32(b, c, m1, 0xB1), m0, 0xE4);
}

// The eight values of one (row, group), as bytes for v_perm_b32: l0 / l1 the low
// bytes of codes 0..3 / 4..7, h0 / h1 the high bytes.
struct ValueTable {
  unsigned l0, l1, h0, h1;
};

// The table of eight 16-bit values, two per word.
__device__ __forceinline__ ValueTable table_of_pairs(const unsigned (&p)[4]) {
  return ValueTable{__builtin_amdgcn_perm(p[1], p[0], 0x06040200u), __builtin_amdgcn_perm(p[3], p[2], 0x06040200u),
                    __builtin_amdgcn_perm(p[1], p[0], 0x07050301u), __builtin_amdgcn_perm(p[3], p[2], 0x07050301u)};
}

template <int XDT>
__device__ __forceinline__ ValueTable value_table(unsigned scale_bits, unsigned zero, int sdt) {
  const float s = sdt == kBF16 ? to_f32<kBF16>(uint16_t(scale_bits)) : to_f32<kF16>(uint16_t(scale_bits));
  const float z = float(zero);
  unsigned p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = s * (float(2 * i) - z), b = s * (float(2 * i + 1) - z);
    if (sdt != XDT) {  // round to the scale's type first, as the restored weight does
      if (sdt == kBF16) round_pair<kBF16>(a, b);
      else round_pair<kF16>(a, b);
    }
    p[i] = round_pair_bits<XDT>(a, b);
  }
  return table_of_pairs(p);
}

// T_s of dequant_word: the code of column 4 n + s in bits 4 n .. 4 n + 2.
template <int S>
__device__ __forceinline__ void code_word(unsigned p0, unsigned p1, unsigned p2, unsigned (&t)[4]) {
  const unsigned M0 = 0x11111111u, M1 = 0x22222222u;
  if constexpr (S == 0) t[0] = select3(p0, p1 << 1, p2 << 2, M0, M1);
  if constexpr (S == 1) t[1] = select3(p0 >> 1, p1, p2 << 1, M0, M1);
  if constexpr (S == 2) t[2] = select3(p0 >> 2, p1 >> 1, p2, M0, M1);
  if constexpr (S == 3) t[3] = select3(p0 >> 3, p1 >> 2, p2 >> 1, M0, M1);
}
__device__ __forceinline__ void code_words(unsigned p0, unsigned p1, unsigned p2, unsigned (&t)[4]) {
  code_word<0>(p0, p1, p2, t);
  code_word<1>(p0, p1, p2, t);
  code_word<2>(p0, p1, p2, t);
  code_word<3>(p0, p1, p2, t);
}

// A operands of steps b = ODD and b = ODD + 2 of one word: element e of step b is
// column 8 b + e.  A quarter (i, h) gives columns 4 h + 2 i and 4 h + 2 i + 1 of both.
template <bool ODD>
__device__ __forceinline__ void expand_quarter(const unsigned (&t)[4], const ValueTable& v, int i, int h, u32x4_t& a0,
                                               u32x4_t& a2) {
  const unsigned both = ODD ? __builtin_amdgcn_bitop3_b32(t[2 * i] >> 8, t[2 * i + 1], 0x00ff00ffu, 0xE4)
                            : __builtin_amdgcn_bitop3_b32(t[2 * i], t[2 * i + 1] << 8, 0x00ff00ffu, 0xE4);
  const unsigned sel = (h ? both >> 4 : both) & 0x07070707u;
  const unsigned lo = __builtin_amdgcn_perm(v.l1, v.l0, sel), hi = __builtin_amdgcn_perm(v.h1, v.h0, sel);
  a0[2 * h + i] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
  a2[2 * h + i] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
}
template <bool ODD>
__device__ __forceinline__ void expand_steps(const unsigned (&t)[4], const ValueTable& v, u32x4_t& a0, u32x4_t& a2) {
#pragma unroll
  for (int q = 0; q < 4; ++q) expand_quarter<ODD>(t, v, q >> 1, q & 1, a0, a2);
}

}  // namespace fx
