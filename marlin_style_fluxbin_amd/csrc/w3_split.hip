// One-row W3 GEMV with the reference's split contract on the matrix cores (inline_main,
// m1_out; csrc/w3_lut.cu:37-189): fp32 partial sums of every groups_per_split groups
// and their sum in split order, in one launch.
//
// What bounded it: the table kernel (w3_lut.hip) makes 48 data-dependent LDS reads per
// row and group, which serialise on banks, and a second launch summed its partials.
// Here a (row, group)'s eight weight values become matrix operands by byte lookup
// (w3_values.h), about two VALU instructions a weight.  Measured (bf16, desc_act,
// decoded_bf16): 12288 x 4096 in 8 splits 10.9 us and 4096 x 12288 in 48 splits 11.4 us
// a launch (two layers' Linears on the observed_exact route, six of these and eight
// one-split launches: 315 -> 110 us).  The bound is the chain of loads, gather and
// expansion of six waves a SIMD (with 92 registers, five waves: 11.2).
//
// Weights.  With a zero-point of 0..7, s (q - z) has at most 14 significant bits (bf16 or
// fp16 scale times an integer of three bits), so it is exactly hi + lo of two bf16 values;
// decoded_bf16 arithmetic drops lo where |q - z| = 3, which is all it needs when every
// zero-point is 3 or 4 (the other products are bf16 numbers): the lo chain runs only for
// structural arithmetic or where a lane sees another zero-point.  fp16 activations are
// split the same way into two columns.  Every product is exact in fp32.
//
// Zero-points above 7 (the entry points take the whole byte; a checked layout has none)
// need up to 19 bits, and a scale that is not finite, or whose products overflow bf16,
// would reach the other splits of its batch as 0 x infinity.  Where a batch holds such a
// (row, group), the row's sums are formed again in fp32, in the table kernel's arithmetic
// (odd_group), after the matrix chain.  The others pay a compare a batch for it: two
// layers' Linears on the observed_exact route take 110.0 us with it and 109.4 without
// (111 with the odd weights' tables zeroed ahead of the chain and their sums added).
//
// A workgroup owns 16 rows; wave w takes the four-group batches w, w + 8, ...  k-block
// l / 16 of an instruction carries group 4 i + l / 16, and column 2 j (+ 1 for the low
// digit of fp16 activations) of the result only sees the groups of the batch's j-th
// split (the other lanes read a zero operand), so one accumulator holds up to four
// splits.  The batches' sums meet in LDS and are added in batch order, then split order.
#include "common.h"
#include "w3_mfma.hip"
#include "w3_split_launch.h"
#include "w3_values.h"

namespace fx {

constexpr int kSplitWaves = 8;

// The tables of the hi and lo halves of one (row, group)'s eight weights.
__device__ __forceinline__ void split_tables(unsigned scale_bits, unsigned zero, int sdt, bool decoded, ValueTable& hi,
                                             ValueTable& lo) {
  const float s = sdt == kBF16 ? to_f32<kBF16>(uint16_t(scale_bits)) : to_f32<kF16>(uint16_t(scale_bits));
  const float z = float(zero);
  unsigned h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float da = float(2 * i) - z, db = float(2 * i + 1) - z;
    float a = s * da, b = s * db, ra = a, rb = b;
    h[i] = round_pair_bits<kBF16>(a, b);
    ra = decoded && fabsf(da) == 3.f ? 0.f : ra - a;
    rb = decoded && fabsf(db) == 3.f ? 0.f : rb - b;
    l[i] = round_pair_bits<kBF16>(ra, rb);
  }
  hi = table_of_pairs(h);
  lo = table_of_pairs(l);
}

// Two bf16 values with infinities and NaN replaced by zero.
__device__ __forceinline__ unsigned finite_pair(unsigned v) {
  const unsigned lo = (v & 0x7f80u) == 0x7f80u ? 0u : v & 0xffffu;
  return lo | ((v & 0x7f800000u) == 0x7f800000u ? 0u : v & 0xffff0000u);
}

// Whether a (row, group)'s weights are not each two bf16 values: |q - z| > 7, or |s| of
// 2^125 and more (bf16: 7 s overflows), infinite or NaN.
__device__ __forceinline__ bool is_odd_group(unsigned scale_bits, unsigned zero, int sdt) {
  return zero > 7u || (scale_bits & 0x7fffu) >= (sdt == kBF16 ? 0x7e00u : 0x7c00u);
}

// One (row, group)'s sum in fp32: s sum (q - z) x, and for decoded arithmetic the
// correction of the weights with |q - z| = 3.  planes: its 16 bytes a plane, from `at` on;
// x: the group's 16 operand units (their low digits `low_units` on, with fp16
// activations).  Rare and small rather than fast: one byte column at a time.
template <int XDT>
__device__ __forceinline__ float odd_group(__amdgpu_buffer_rsrc_t planes, int at, int plane_stride, const u32x4_t* x,
                                           int low_units, unsigned scale_bits, unsigned zero, int sdt, bool decoded) {
  float dot = 0.f, three = 0.f;
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const u32x4_t hi = x[c];
    u32x4_t lo = {0u, 0u, 0u, 0u};
    if constexpr (XDT == kF16) lo = x[low_units + c];
    unsigned b[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) b[p] = __builtin_amdgcn_raw_buffer_load_b8(planes, at + c, p * plane_stride, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int shift = 16 * (j & 1);
      const float v = to_f32<kBF16>(uint16_t(hi[j >> 1] >> shift)) + to_f32<kBF16>(uint16_t(lo[j >> 1] >> shift));
      const int q = int(((b[0] >> j) & 1u) | (((b[1] >> j) & 1u) << 1) | (((~b[2] >> j) & 1u) << 2)), d = q - int(zero);
      dot += float(d) * v;
      if (d == 3) three += v;
      if (d == -3) three -= v;
    }
  }
  const float s = sdt == kBF16 ? to_f32<kBF16>(uint16_t(scale_bits)) : to_f32<kF16>(uint16_t(scale_bits));
  float sum = dot * s;
  if (decoded) sum += three * (round_to<kBF16>(3.f * s) - 3.f * s);
  return sum;
}

// Elements 8 i .. 8 i + 7 of a 16-bit array.
__device__ __forceinline__ u32x4_t load_eight(const uint16_t* p, int i, int aligned) {
  if (aligned) return reinterpret_cast<const u32x4_t*>(p)[i];
  u32x4_t v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = unsigned(p[8 * i + 2 * j]) | (unsigned(p[8 * i + 2 * j + 1]) << 16);
  return v;
}

template <int XDT>
__global__ __launch_bounds__(kSplitWaves * 64, 6) void w3_split_kernel(SplitArgs a) {
  extern __shared__ u32x4_t split_lds[];
  __shared__ int nonfinite;  // an activation is infinite or NaN
  if (threadIdx.x == 0) nonfinite = 0;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int r = lane & 15, kb = lane >> 4, c = lane & 15;
  const int batches = (a.G + 3) >> 2, K = a.G * 128;
  const int row0 = xcd_local_index8(blockIdx.x, gridDim.x) * 16;
  // LDS: the operands [digit][batches x 64 units], 16 units of zeros, the batches' sums
  // [batch][slot][16], the activations in their own order (with a permutation)
  constexpr int kDigits = XDT == kF16 ? 2 : 1;
  const int units = batches * 64;
  u32x4_t* xs = split_lds;
  u32x4_t* zero16 = xs + kDigits * units;
  float* sums = reinterpret_cast<float*>(zero16 + 16);
  const int slots = 4 >> a.slot_shift;  // splits in a batch
  uint16_t* raw = reinterpret_cast<uint16_t*>(sums + batches * slots * 16);

  // ---- activations and their columns first (the wave's loads complete in order, and
  // staging needs only these), then the weights of the wave's first batch
  constexpr int kTurns = kSplitMaxColumns / 8 / (kSplitWaves * 64);
  u32x4_t xv[kTurns], pv[kTurns];
#pragma unroll
  for (int k = 0; k < kTurns; ++k) {
    const int i = int(threadIdx.x) + k * (kSplitWaves * 64);
    if (i < K / 8) {
      xv[k] = load_eight(a.x, i, a.x16);
      if (a.perm) pv[k] = load_eight(reinterpret_cast<const uint16_t*>(a.perm), i, a.perm16);
    }
  }
  const int row = min(row0 + r, a.O - 1);
  const unsigned go = unsigned(a.G) * unsigned(a.O);
  const auto rp = buffer_resource_2g(a.planes, go * 48u);
  const auto rs = buffer_resource_2g(a.scales, go * 2u);
  const auto rz = buffer_resource_2g(a.zeros ? (const void*)a.zeros : (const void*)a.scales, a.zeros ? go : 0u);
  const unsigned zero_default = a.zeros ? 0u : 4u;  // absent zero-points read as 0
  struct Loads {
    u32x4_t p[3];
    unsigned s, z;
  };
  const auto plane_offset = [&](int batch) { return (4 * batch * 3 * a.O + lane_times_rows(kb, 3 * a.O) + row) * 16; };
  auto issue = [&](int batch, Loads& L) __attribute__((always_inline)) {
    const int out = batch < batches && 4 * batch + kb < a.G ? 0 : kOutOfRange;  // zero scales: zero weights
    const int e = 4 * batch * a.O + lane_times_rows(kb, a.O) + row;
    const int off = plane_offset(batch) | out;
    L.s = __builtin_amdgcn_raw_buffer_load_b16(rs, (e * 2) | out, 0, 0);
    L.z = __builtin_amdgcn_raw_buffer_load_b8(rz, e | out, 0, 0);
#pragma unroll
    for (int p = 0; p < 3; ++p) L.p[p] = load_b128_stream(rp, off, p * a.O * 16);
  };
  Loads next;
  issue(wave, next);

  // ---- activations in the payload's order, as bf16 operands; columns past K are zero
  if (threadIdx.x < 16) zero16[threadIdx.x] = u32x4_t{0u, 0u, 0u, 0u};
  if (a.perm) {
#pragma unroll
    for (int k = 0; k < kTurns; ++k) {
      const int i = int(threadIdx.x) + k * (kSplitWaves * 64);
      if (i < K / 8) reinterpret_cast<u32x4_t*>(raw)[i] = xv[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTurns; ++k) {
    const int u = int(threadIdx.x) + k * (kSplitWaves * 64);
    if (u >= units) break;
    unsigned v[4] = {0u, 0u, 0u, 0u};
    if (u < K / 8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {  // entries outside [0, K) read zero
        const int lo = int(int16_t(pv[k][j])), hi = int(pv[k][j]) >> 16;
        v[j] = !a.perm ? xv[k][j]
                       : (unsigned(lo) < unsigned(K) ? raw[lo] : 0u) | ((unsigned(hi) < unsigned(K) ? raw[hi] : 0u) << 16);
      }
    }
    u32x4_t hi, lo;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (XDT == kBF16) {
        hi[j] = v[j];
      } else {
        float f0 = to_f32<kF16>(uint16_t(v[j])), f1 = to_f32<kF16>(uint16_t(v[j] >> 16)), h0 = f0, h1 = f1;
        hi[j] = round_pair_bits<kBF16>(h0, h1);
        f0 = fabsf(f0) < INFINITY ? f0 - h0 : 0.f;  // 11 bits = 8 + 3: exact; an infinity or NaN has no low digit
        f1 = fabsf(f1) < INFINITY ? f1 - h1 : 0.f;
        lo[j] = round_pair_bits<kBF16>(f0, f1);
      }
    }
    bool odd = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) odd |= finite_pair(hi[j]) != hi[j];
    if (odd) nonfinite = 1;
    xs[u] = hi;
    if constexpr (XDT == kF16) xs[units + u] = lo;
  }
  __syncthreads();

  // ---- this lane's operand: column c = 2 slot + digit, its own split's groups
  const int slot = kb >> a.slot_shift;
  const int digit = c & 1;
  const bool active = (c >> 1) == slot && digit < kDigits;
  unsigned long long any_odd = 0;  // lanes with an odd group in one of the wave's batches
  for (int batch = wave; batch < batches; batch += kSplitWaves) {
    const Loads cur = next;
    issue(batch + kSplitWaves, next);
    const unsigned zero = (cur.z & 0xffu) | zero_default;
    any_odd |= __builtin_amdgcn_ballot_w64(is_odd_group(cur.s, zero, a.sdt));
    ValueTable hi, lo;
    split_tables(cur.s, zero, a.sdt, a.decoded, hi, lo);
    const bool low = !a.decoded || __builtin_amdgcn_ballot_w64(zero != 3u && zero != 4u && 4 * batch + kb < a.G) != 0;
    const u32x4_t* src = active ? xs + digit * units + batch * 64 + kb * 16 : zero16;
    f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      unsigned t[4];
      code_words(cur.p[0][w], cur.p[1][w], cur.p[2][w], t);
#pragma unroll
      for (int odd = 0; odd < 2; ++odd) {  // two steps at a time: the registers of six waves a SIMD
        u32x4_t B[2] = {src[4 * w + odd], src[4 * w + odd + 2]}, A[2];
        const auto multiply = [&](const ValueTable& table) __attribute__((always_inline)) {
          if (odd) expand_steps<true>(t, table, A[0], A[1]);
          else expand_steps<false>(t, table, A[0], A[1]);
#pragma unroll
          for (int b = 0; b < 2; ++b)
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, A[b]),
                                                        __builtin_bit_cast(bf16x8_t, B[b]), d, 0, 0, 0);
        };
        multiply(hi);
        if (low) {  // wave-uniform
          // an infinity's product is the hi half's alone (0 x infinity would make it NaN)
          if (nonfinite) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int j = 0; j < 4; ++j) B[b][j] = finite_pair(B[b][j]);
          }
          multiply(lo);
        }
      }
    }
    // lane (c, kb) holds rows 4 kb .. + 3 of column c; column 2 j (+ 1) is split j
    if constexpr (XDT == kF16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] += dpp_move<kDppXor1>(d[j]);
    }
    if (digit == 0 && (c >> 1) < slots) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sums[(batch * slots + (c >> 1)) * 16 + 4 * kb + j] = d[j];
    }
  }
  // ---- odd groups: the sums of their rows in their batches, formed again
  for (int batch = wave; any_odd != 0 && batch < batches; batch += kSplitWaves) {
    Loads L;
    issue(batch, L);
    const unsigned zero = (L.z & 0xffu) | zero_default;
    const unsigned long long odd = __builtin_amdgcn_ballot_w64(is_odd_group(L.s, zero, a.sdt));
    if (((odd | odd >> 16 | odd >> 32 | odd >> 48) >> r) & 1u) {  // this lane's row has one
      float sum = 0.f;
      if (4 * batch + kb < a.G)
        sum = odd_group<XDT>(rp, plane_offset(batch), a.O * 16, xs + batch * 64 + kb * 16, units, L.s, zero, a.sdt, a.decoded);
      float* at = sums + (batch * slots + slot) * 16 + r;
#pragma unroll 1
      for (int k = 0; k < 4; ++k) {  // the groups in turn; a split's first one starts its sum
        wave_lds_order();
        if (kb == k) *at = k == slot << a.slot_shift ? sum : *at + sum;
      }
    }
  }
  __syncthreads();

  // ---- partials in batch order (over the batches' sums), the output in split order;
  // eight LDS reads in flight, added in order
  const int splits = (a.G + a.gps - 1) / a.gps;
  const int per = slots > 1 ? 1 : (min(a.gps, a.G) + 3) / 4;  // batches of a split
  const int col = int(threadIdx.x & 15), o = row0 + col;
  const auto total = [&](int first, int last) {
    float t = 0.f;
    for (int i = first; i < last; i += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = i + j < last ? sums[(i + j) * 16 + col] : 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (i + j < last) t += v[j];
    }
    return t;
  };
  if (a.partial || per > 1) {
    float mine[4];  // at most 128 splits over 32 threads a row
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int s = int(threadIdx.x >> 4) + k * (kSplitWaves * 4);
      mine[k] = s < splits ? total(s * per, min((s + 1) * per, batches * slots)) : 0.f;
      if (a.partial && s < splits && o < a.O) a.partial[size_t(s) * a.O + o] = mine[k];
    }
    if (a.out && per > 1) {
      __syncthreads();  // every batch's sums have been read
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = int(threadIdx.x >> 4) + k * (kSplitWaves * 4);
        if (s < splits) sums[s * 16 + col] = mine[k];
      }
      __syncthreads();
    }
  }
  if (a.out && threadIdx.x < 16 && o < a.O) a.out[o] = from_f32<XDT>(total(0, splits));
}

void launch_split(int xdt, SplitArgs a, hipStream_t s) {
  a.slot_shift = a.gps >= 4 || a.gps >= a.G ? 2 : a.gps - 1;
  const int batches = (a.G + 3) / 4, slots = 4 >> a.slot_shift;
  const size_t lds = size_t(batches) * 1024 * (xdt == kF16 ? 2 : 1) + 256 + size_t(batches) * slots * 64 +
                     (a.perm ? size_t(a.G) * 256 : 0);
  const dim3 grid(unsigned((a.O + 15) / 16)), block(kSplitWaves * 64);
  if (lds > 65536) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(xdt == kBF16 ? &w3_split_kernel<kBF16> : &w3_split_kernel<kF16>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
  }
  if (xdt == kBF16)
    hipLaunchKernelGGL(w3_split_kernel<kBF16>, grid, block, lds, s, a);
  else
    hipLaunchKernelGGL(w3_split_kernel<kF16>, grid, block, lds, s, a);
}

}  // namespace fx
