// W3 GEMM for many activation rows: 48 NW output rows by 16 MT activation rows a
// workgroup, everything staged through LDS by the memory pipeline itself.
//
// What bounds it: with a hundred and more rows per weight the matrix cores do, if the
// operands arrive.  The kernel of w3_gemm.h reads every activation operand once per
// wave; here NW consumer waves (three 16-row tiles each) share them.  Two producer
// waves issue buffer loads that write LDS directly (no registers, so the prefetch is as
// deep as LDS allows): the packed activations of one half-word (two steps) into a ring
// of kSlots slots, D - 1 half-words ahead, and the plane rows of the next batch into
// the other of two buffers.  Consumers never wait for global memory but for their
// rows' scales and zero-points, a batch ahead.
//
// Order.  Barrier n is passed when the activations of half-word n + 1 (and the planes
// issued before them) have landed: the producers wait with a counted vmcnt.  Between
// barriers n and n + 1 a consumer multiplies half-word n and starts reading half-word
// n + 1, so its LDS reads always have a step's matrix instructions to arrive, and a
// slot is written again two barriers after its last read was used.  The barrier is the
// bare instruction: its waits are the ones stated here.
//
// The expansion of half-word n + 1 (w3_values.h) runs between the matrix instructions
// of half-word n, in pieces of about a dozen instructions that scheduling barriers keep
// in place: left to the scheduler they gathered at one end, and the matrix cores idled.
//
// Measured (bf16, 12288 x 4096): 512 rows 55.3 us against 68.4 for the other kernel's
// 4 x 8 tiles and 79 for the restored weight's library product with its restore; the
// main loop multiplies at 12.2 ns per matrix instruction and SIMD, what a large library
// product (1.41 PFLOP/s) reaches on this card.
#pragma once
#include "w3_gemm.h"

namespace fx {

constexpr int kTallAhead = 4;  // D: half-words in flight or being read
constexpr int kTallSlots = 5;
constexpr int kTallProducers = 2;

// All memory operations of the wave stay on their side of it.
__device__ __forceinline__ void ordered_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Wait until at most N vector memory operations of the wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, u32x4_t* lds, int voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voffset, 0, 0, 0);
}

template <int XDT, int MT, int NW>
__global__ __launch_bounds__((NW + kTallProducers) * 64) void w3_gemm_tall_kernel(GemmArgs a) {
  constexpr int RT = kTallTiles, D = kTallAhead, S = kTallSlots, PP = kTallProducers;
  constexpr int SLOT = 2 * MT * 64;             // 16-byte units of a half-word
  constexpr int PLANES = NW * RT * 3 * 64;      // of a batch's plane rows: [tile][plane][lane]
  constexpr int XL = 2 * MT / PP;               // loads of a half-word per producer
  constexpr int WL = NW * RT * 3 / PP, WS = WL / 3;  // of a batch's planes; in each of three steps
  static_assert(2 * MT % PP == 0 && NW * RT * 3 % (PP * 3) == 0, "producers share the loads evenly");
  static_assert(D == 4 && S == D + 1, "the waits and the slot reuse below are for this depth");
  __shared__ u32x4_t ring[S * SLOT];
  __shared__ u32x4_t planes[2 * PLANES];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int r = lane & 15, kb = lane >> 4;
  // row blocks of one output block run on one XCD, next to each other: they share its weights
  const int linear = xcd_local_index8(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int row0 = linear / int(gridDim.y) * (16 * RT * NW);
  const int block = linear % int(gridDim.y), m0 = block * 16 * MT;
  const int batches = (a.G + 3) >> 2;
  const int b0 = int(blockIdx.z) * a.batches_per_split;
  const int b1 = min(batches, b0 + a.batches_per_split);
  const int plane_stride = a.O * 16;
  const unsigned go = unsigned(a.G) * unsigned(a.O);

  if (wave >= NW) {
    const int p = wave - NW;
    const unsigned packed_bytes = unsigned(batches) * (16u * MT * 1024u);
    const auto rx = buffer_resource_2g(reinterpret_cast<const char*>(a.packed) + size_t(block) * packed_bytes, packed_bytes);
    const auto rp = buffer_resource_2g(a.planes, go * 48u);
    const int end = b1 * (16 * MT * 1024);
    // half-word n of the split: steps 4 (h / 2) + h % 2 and two on, [step][MT] operands
    // of 1 KB each; producer p takes step j = p (MT loads).  Past the range: no access.
    auto load_x = [&](int n) __attribute__((always_inline)) {
      const int h = n & 7, base = ((b0 + (n >> 3)) * 16 + 4 * (h >> 1) + (h & 1)) * (MT * 1024);
      u32x4_t* dst = ring + (unsigned(n) % S) * SLOT;
#pragma unroll
      for (int i = 0; i < XL; ++i) {
        const int unit = p * XL + i, j = unit / MT, mt = unit % MT;
        const int off = base + (2 * j * MT + mt) * 1024;
        load_to_lds(rx, dst + unit * 64, off < end ? off + lane * 16 : kOutOfRange);
      }
    };
    // third `part` of the plane rows of batch b: [tile][plane], lane (r, kb) the 16 bytes
    // of row r of the tile in group 4 b + kb (rows past O: row O - 1, never stored)
    auto load_w = [&](int b, int part) __attribute__((always_inline)) {
      const int out = b < b1 && 4 * b + kb < a.G ? 0 : kOutOfRange;
      u32x4_t* dst = planes + ((b - b0) & 1) * PLANES;
#pragma unroll
      for (int i = 0; i < WS; ++i) {
        const int unit = p * WL + part * WS + i, tile = unit / 3, plane = unit % 3;
        const int row = min(row0 + 16 * tile + r, a.O - 1);
        const int off = (4 * b * 3 * a.O + lane_times_rows(kb, 3 * a.O) + row) * 16 + plane * plane_stride;
        load_to_lds(rp, dst + unit * 64, off | out);
      }
    };
#pragma unroll
    for (int part = 0; part < 3; ++part) load_w(b0, part);
#pragma unroll
    for (int n = 0; n < D - 1; ++n) load_x(n);
    int n = 0;
    for (int b = b0; b < b1; ++b) {
#pragma unroll
      for (int h = 0; h < 8; ++h, ++n) {
        if (h < 3) load_w(b + 1, h);
        load_x(n + D - 1);
        // outstanding after half-word n + 1: the loads of this step and the D - 3 before
        constexpr int kSteps = D - 2;
        if (h == 0) wait_vmcnt<kSteps * XL + WS>();
        else if (h <= 2) wait_vmcnt<kSteps * XL + 2 * WS>();
        else if (h == 3) wait_vmcnt<kSteps * XL + WS>();
        else wait_vmcnt<kSteps * XL>();
        ordered_barrier();
      }
    }
    wait_vmcnt<0>();  // nothing writes this workgroup's LDS after its last wave has left
    return;
  }

  const auto rs = buffer_resource_2g(a.scales, go * 2u);
  const auto rz = buffer_resource_2g(a.zeros ? (const void*)a.zeros : (const void*)a.scales, a.zeros ? go : 0u);
  const unsigned zero_default = a.zeros ? 0u : 4u;  // absent zero-points read as 0
  const int tile0 = row0 + wave * 16 * RT;
  unsigned sn[RT], zn[RT];
  auto load_scales = [&](int b) __attribute__((always_inline)) {
    const int out = b < b1 && 4 * b + kb < a.G ? 0 : kOutOfRange;  // zero scales: zero weights
#pragma unroll
    for (int tt = 0; tt < RT; ++tt) {
      const int e = 4 * b * a.O + lane_times_rows(kb, a.O) + min(tile0 + 16 * tt + r, a.O - 1);
      sn[tt] = __builtin_amdgcn_raw_buffer_load_b16(rs, (e * 2) | out, 0, 0);
      zn[tt] = __builtin_amdgcn_raw_buffer_load_b8(rz, e | out, 0, 0);
    }
  };
  f32x4_t acc[RT][MT];
#pragma unroll
  for (int tt = 0; tt < RT; ++tt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[tt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  ValueTable tab[RT];
  unsigned pw[RT][3], t[RT][4];  // a word's plane bits, and its codes
  u32x4_t A[2][2][RT];           // the weights of half-word h in A[h % 2]
  u32x4_t B[MT];
  auto tables = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int tt = 0; tt < RT; ++tt) tab[tt] = value_table<XDT>(sn[tt], (zn[tt] & 0xffu) | zero_default, a.sdt);
  };
  auto read_planes = [&](int b, int w) __attribute__((always_inline)) {
    const unsigned* src = reinterpret_cast<const unsigned*>(planes + ((b - b0) & 1) * PLANES + wave * RT * 3 * 64 + lane) + w;
#pragma unroll
    for (int tt = 0; tt < RT; ++tt)
#pragma unroll
      for (int p = 0; p < 3; ++p) pw[tt][p] = src[tt * 768 + p * 256];
  };
  // quarter q (0..3) of the expansion of one tile's half-word of parity `odd`: an even
  // half-word first forms the word's codes
  auto expand = [&](int odd, int tt, int q) __attribute__((always_inline)) {
    if (!odd) {
      if (q == 0) code_word<0>(pw[tt][0], pw[tt][1], pw[tt][2], t[tt]), code_word<1>(pw[tt][0], pw[tt][1], pw[tt][2], t[tt]);
      if (q == 1) code_word<2>(pw[tt][0], pw[tt][1], pw[tt][2], t[tt]);
      if (q == 2) code_word<3>(pw[tt][0], pw[tt][1], pw[tt][2], t[tt]);
    }
    const int i = q >> 1, h = q & 1;
    if (odd) expand_quarter<true>(t[tt], tab[tt], i, h, A[1][0][tt], A[1][1][tt]);
    else expand_quarter<false>(t[tt], tab[tt], i, h, A[0][0][tt], A[0][1][tt]);
  };
  load_scales(b0);
  ordered_barrier();  // barrier 0: the first batch's planes, half-words 0 and 1
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) B[mt] = ring[mt * 64 + lane];
  read_planes(b0, 0);
  tables();
  load_scales(b0 + 1);
#pragma unroll
  for (int u = 0; u < 4 * RT; ++u) expand(0, u >> 2, u & 3);
  int slot = 0;
  for (int b = b0; b < b1; ++b) {
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const int after = slot + 1 == S ? 0 : slot + 1;
      const u32x4_t* here = ring + slot * SLOT + lane;
      const u32x4_t* there = ring + after * SLOT + lane;
      // the next word's planes, a half-word ahead of their codes (the next batch's
      // first: its planes landed by barrier 4)
      if ((h & 1) == 0) {
        if (h < 6) read_planes(b, (h >> 1) + 1);
        else read_planes(b + 1, 0);
      }
      if (h == 7) {
        tables();
        load_scales(b + 2);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int tt = 0; tt < RT; ++tt) acc[tt][mt] = mfma16<XDT>(A[h & 1][j][tt], B[mt], acc[tt][mt]);
          B[mt] = j == 0 ? here[(MT + mt) * 64] : there[mt * 64];
          // a share of half-word h + 1's expansion under these matrix instructions
          const int u0 = (j * MT + mt) * 4 * RT / (2 * MT), u1 = (j * MT + mt + 1) * 4 * RT / (2 * MT);
#pragma unroll
          for (int u = u0; u < u1; ++u) expand((h + 1) & 1, u >> 2, u & 3);
        }
      slot = after;
      if (h < 7 || b + 1 < b1) ordered_barrier();
    }
  }
  gemm_store<XDT, RT, MT>(a, acc, tile0, m0, r, kb);
}

template <int XDT, int MT, int NW>
bool gemm_tall_launch(const GemmPlan& p, const GemmArgs& a, hipStream_t s) {
  const dim3 grid(unsigned((a.O + 16 * kTallTiles * NW - 1) / (16 * kTallTiles * NW)),
                  unsigned((a.M + 16 * MT - 1) / (16 * MT)), unsigned(p.splits));
  hipLaunchKernelGGL((w3_gemm_tall_kernel<XDT, MT, NW>), grid, dim3((NW + kTallProducers) * 64), 0, s, a);
  return true;
}

}  // namespace fx
