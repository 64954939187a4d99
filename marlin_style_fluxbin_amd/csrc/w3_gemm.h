// W3 g128 planar GEMM for gfx950: out[M, O] = x[M, K] . W^T with the dense fallback's
// weight W = round_x(round_scale(s (q - z))) formed in registers, so no [O, K]
// weight is written or read.
//
// Why: for a few to a few hundred rows the product reads each weight once or
// twice, and restoring it to HBM first (2 O K bytes written, 2 O K read back by a
// library product, against 3 O K / 8 of codes) was most of the time.
//
// Exact weights without arithmetic per weight: a (row, group) has eight possible
// values, so each lane forms those eight once per 128 columns, rounded as the
// restore kernel rounds them, and keeps their low and high bytes in two register
// pairs.  v_perm_b32 is then an eight-entry byte lookup with four codes a
// register: two lookups give the low and high bytes of four weights and two more
// byte permutes pair them, about 2.2 VALU instructions per weight in all against
// the 16-bit MFMA operands the restored weight would give, bit for bit.
//
// Operands (v_mfma_f32_16x16x32_{bf16,f16}): lane l holds A[l % 16][8 (l / 16) + j]
// (weights of 16 output rows), B[8 (l / 16) + j][l % 16] (16 activation rows) and
// D[4 (l / 16) + j][l % 16].  k-block l / 16 carries group 4 i + l / 16 of a batch
// of four groups, so a lane's share of a batch is one 16-byte load per plane; the
// weights already carry their scales, so one accumulator serves all groups.
// Step (w, b) of a batch multiplies columns 32 w + 8 b .. + 7 of each group.
//
// Work split: a workgroup owns 16 RT output rows, 16 MT activation rows and a K
// range whose batches its NK waves take in turn; their sums meet in LDS, pairwise.  No
// two waves of a workgroup read the same weights or activations, so nothing is staged:
// gemm_pack_kernel has laid the activations out in operand order (and in the payload's
// column order) once, and every B operand is one coalesced 16-byte load per lane, issued
// PD half-words (two steps each) ahead.  K splits over workgroups leave fp32 partials
// for gemm_finish_kernel, in split order.
#pragma once
#include "w3_gemm_launch.h"
#include "w3_mfma.hip"
#include "w3_values.h"

namespace fx {

template <int XDT>
__device__ __forceinline__ f32x4_t mfma16(const u32x4_t& a, const u32x4_t& b, const f32x4_t& d) {
  if constexpr (XDT == kBF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), d,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), d, 0,
                                                  0, 0);
}

// A wave's outputs (or its split's partials).
template <int XDT, int RT, int MT>
__device__ __forceinline__ void gemm_store(const GemmArgs& a, const f32x4_t (&acc)[RT][MT], int row0, int m0, int r,
                                           int kb) {
  // lane (r, kb): rows 4 kb .. + 3 of each tile, activation row m0 + 16 mt + r
#pragma unroll
  for (int tt = 0; tt < RT; ++tt) {
    const int o = row0 + 16 * tt + 4 * kb;
    if (o >= a.O) continue;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.bias && !a.partial) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (o + j < a.O) bias[j] = to_f32<XDT>(a.bias[o + j]);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = m0 + 16 * mt + r;
      if (m >= a.M) continue;
      const f32x4_t d = acc[tt][mt];
      if (a.partial) {
        float* dst = a.partial + (size_t(blockIdx.z) * a.M + m) * a.O + o;
        if (a.vec) {
          *reinterpret_cast<f32x4_t*>(dst) = d;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (o + j < a.O) dst[j] = d[j];
        }
      } else {
        uint16_t* dst = a.out + size_t(m) * a.O + o;
        uint16_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = from_f32<XDT>(d[j] + bias[j]);
        if (a.vec) {
          *reinterpret_cast<uint2*>(dst) =
              uint2{unsigned(v[0]) | (unsigned(v[1]) << 16), unsigned(v[2]) | (unsigned(v[3]) << 16)};
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (o + j < a.O) dst[j] = v[j];
        }
      }
    }
  }
}

template <int XDT, int RT, int MT, int NK, int PD, bool NEXT>
__global__ __launch_bounds__(NK * 64) void w3_gemm_kernel(GemmArgs a) {
  __shared__ f32x4_t red[NK > 1 ? NK / 2 * RT * MT * 64 : 1];
  const int lane = threadIdx.x & 63, part = wave_index();
  const int r = lane & 15, kb = lane >> 4;
  const int row0 = xcd_local_index8(blockIdx.x, gridDim.x) * (16 * RT);
  const int m0 = int(blockIdx.y) * 16 * MT;
  const int batches = (a.G + 3) >> 2;
  const int b0 = int(blockIdx.z) * a.batches_per_split;
  const int b1 = min(batches, b0 + a.batches_per_split);

  const unsigned go = unsigned(a.G) * unsigned(a.O);
  const auto rp = buffer_resource_2g(a.planes, go * 48u);
  const auto rs = buffer_resource_2g(a.scales, go * 2u);
  const auto rz = buffer_resource_2g(a.zeros ? (const void*)a.zeros : (const void*)a.scales, a.zeros ? go : 0u);
  const unsigned zero_default = a.zeros ? 0u : 4u;  // absent zero-points read as 0
  // packed activations of this block of rows: [batch][step][MT][lane] units
  const unsigned packed_bytes = unsigned(batches) * (16u * MT * 1024u);
  const auto rx = buffer_resource_2g(reinterpret_cast<const char*>(a.packed) + size_t(blockIdx.y) * packed_bytes,
                                     packed_bytes);
  int prow[RT];  // rows past O read row O - 1 (never stored)
#pragma unroll
  for (int tt = 0; tt < RT; ++tt) prow[tt] = min(row0 + 16 * tt + r, a.O - 1);
  const int plane_stride = a.O * 16;
  struct Loads {
    u32x4_t p[RT][3];
    unsigned s[RT], z[RT];
  };
  auto issue = [&](int batch, Loads& L) __attribute__((always_inline)) {
    // batches past the range and groups past G read zeros: a zero scale, so zero weights
    const int out = batch < b1 && 4 * batch + kb < a.G ? 0 : kOutOfRange;  // the sign bit: past the end
    const int gb = batch * 4;
#pragma unroll
    for (int tt = 0; tt < RT; ++tt) {
      const int e = gb * a.O + lane_times_rows(kb, a.O) + prow[tt];
      const int poff = ((gb * 3 * a.O + lane_times_rows(kb, 3 * a.O) + prow[tt]) * 16) | out;
      L.s[tt] = __builtin_amdgcn_raw_buffer_load_b16(rs, (e * 2) | out, 0, 0);
      L.z[tt] = __builtin_amdgcn_raw_buffer_load_b8(rz, e | out, 0, 0);
      L.p[tt][0] = load_b128_stream(rp, poff, 0);
      L.p[tt][1] = load_b128_stream(rp, poff, plane_stride);
      L.p[tt][2] = load_b128_stream(rp, poff, 2 * plane_stride);
    }
  };
  // B operands of half-word h (0..7) of a batch: steps 4 (h / 2) + h % 2 and two on
  u32x4_t B[PD + 1][2][MT];
  const int voff = lane * 16;
  auto fetch = [&](int slot, int batch, int h) __attribute__((always_inline)) {
    const int base = batch < b1 ? batch * (16 * MT * 1024) : int(packed_bytes);  // past the end: zeros, unused
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        B[slot][j][mt] = load_b128(rx, voff + base + ((4 * (h >> 1) + (h & 1) + 2 * j) * MT + mt) * 1024, 0);
  };
  f32x4_t acc[RT][MT];
#pragma unroll
  for (int tt = 0; tt < RT; ++tt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[tt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  static_assert(PD < 8 && 8 % (PD + 1) == 0, "the operand ring must divide a batch");
  Loads next;
  int batch = b0 + part;
  issue(batch, next);
#pragma unroll
  for (int h = 0; h < PD; ++h) fetch(h, batch, h);
  __builtin_amdgcn_sched_barrier(0);
  for (; batch < b1; batch += NK) {
    if (!NEXT && batch != b0 + part) issue(batch, next);
    const Loads cur = next;
    ValueTable tab[RT];
#pragma unroll
    for (int tt = 0; tt < RT; ++tt)
      tab[tt] = value_table<XDT>(cur.s[tt], (cur.z[tt] & 0xffu) | zero_default, a.sdt);
    if (NEXT && batch + NK < b1) issue(batch + NK, next);
    unsigned t[RT][4];
    u32x4_t A[2][2][RT];  // the weights of half-word h in A[h % 2]
    auto expand = [&](int h) __attribute__((always_inline)) {
      const int w = h >> 1;
#pragma unroll
      for (int tt = 0; tt < RT; ++tt) {
        if ((h & 1) == 0) code_words(cur.p[tt][0][w], cur.p[tt][1][w], cur.p[tt][2][w], t[tt]);
        if (h & 1) expand_steps<true>(t[tt], tab[tt], A[1][0][tt], A[1][1][tt]);
        else expand_steps<false>(t[tt], tab[tt], A[0][0][tt], A[0][1][tt]);
      }
    };
    expand(0);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const int ahead = h + PD;
      fetch(ahead % (PD + 1), batch + (ahead >> 3) * NK, ahead & 7);
      __builtin_amdgcn_sched_barrier(0);
      // the next half-word's expansion runs between this one's matrix instructions
      if (h < 7) expand(h + 1);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int tt = 0; tt < RT; ++tt)
            acc[tt][mt] = mfma16<XDT>(A[h & 1][j][tt], B[h % (PD + 1)][j][mt], acc[tt][mt]);
#pragma unroll
      for (int i = 0; i < 2 * RT * MT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                        // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (20 + MT - 1) / MT, 0);       // its share of the expansion
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the waves' sums, pairwise: wave p adds wave p + n for n = NK / 2, NK / 4, ..., 1
  static_assert((NK & (NK - 1)) == 0, "waves per workgroup must be a power of two");
#pragma unroll
  for (int n = NK / 2; n > 0; n >>= 1) {
    f32x4_t* slot = red + (part & (n - 1)) * (RT * MT * 64) + lane;
    if (part >= n && part < 2 * n) {
#pragma unroll
      for (int tt = 0; tt < RT; ++tt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) slot[(tt * MT + mt) * 64] = acc[tt][mt];
    }
    __syncthreads();
    if (part < n) {
#pragma unroll
      for (int tt = 0; tt < RT; ++tt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[tt][mt] += slot[(tt * MT + mt) * 64];
    }
    __syncthreads();
  }
  if (part > 0) return;
  gemm_store<XDT, RT, MT>(a, acc, row0, m0, r, kb);
}

template <int XDT, int RT, int MT, int NK, int PD, bool NEXT>
bool gemm_launch(const GemmPlan& p, const GemmArgs& a, hipStream_t s) {
  const dim3 grid(unsigned((a.O + 16 * RT - 1) / (16 * RT)), unsigned((a.M + 16 * MT - 1) / (16 * MT)),
                  unsigned(p.splits));
  hipLaunchKernelGGL((w3_gemm_kernel<XDT, RT, MT, NK, PD, NEXT>), grid, dim3(NK * 64), 0, s, a);
  return true;
}

}  // namespace fx
