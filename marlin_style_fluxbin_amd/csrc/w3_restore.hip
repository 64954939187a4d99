// Dequantize a W3 payload to a dense [O,K] weight with the reference's rounding points
// (restore_planar_w3, gptq_deployment.py:247-260): round_scale_dtype(s*(q-z)),
// then round to the weight dtype.  Sorted column s = 128g+8c+j of row o lands
// at weight[o, perm[s]].
//
// Bound by the store of 2 O K bytes.  A lane expands one 32-bit word of a row's three
// plane rows (32 columns) through the (row, group)'s value table (w3_values.h), about
// three VALU instructions a weight where the bit-by-bit expansion took fourteen and was
// the bound: 12288 x 4096 identity order 34.6 -> 25.9 us (43.1 -> 35.8 with a
// permutation), 4096 x 4096 13.9 -> 8.8 (16.1 -> 13.4); a fill of the 100 MB takes 17.8.
#include "common.h"
#include "w3_restore_launch.h"
#include "w3_values.h"

namespace fx {

// What one lane loads of word w of row o, group g, and its 32 columns as four 16-byte
// vectors in column order.
struct RestoreWord {
  unsigned p[3], scale, zero;
};
__device__ __forceinline__ RestoreWord load_word(const RestoreArgs& a, int g, int o, int w) {
  const size_t go = size_t(g) * a.O + o, plane = size_t(a.O) * 16;
  const uint8_t* row = a.planes + size_t(g) * 3 * plane + size_t(o) * 16 + 4 * w;
  return {{*reinterpret_cast<const unsigned*>(row), *reinterpret_cast<const unsigned*>(row + plane),
           *reinterpret_cast<const unsigned*>(row + 2 * plane)},
          a.scales[go],
          a.zeros ? a.zeros[go] : 4u};
}
template <int WDT>
__device__ __forceinline__ void restore_word(const RestoreWord& in, int sdt, u32x4_t (&v)[4]) {
  const ValueTable table = value_table<WDT>(in.scale, in.zero, sdt);
  unsigned t[4];
  code_words(in.p[0], in.p[1], in.p[2], t);
  expand_steps<false>(t, table, v[0], v[2]);
  expand_steps<true>(t, table, v[1], v[3]);
}

// Identity order.  A wave owns 16 rows and kWaveGroups consecutive groups, four lanes
// to a row of a group, every load issued ahead; the vectors pass through the wave's own
// LDS so that a row's 512 bytes leave together (element stores when the weight is not
// 16-byte aligned).
constexpr int kWaveGroups = kRestoreGroups / 4;
template <int WDT>
__global__ __launch_bounds__(256) void w3_restore_kernel(RestoreArgs a) {
  constexpr int kRow = 16 * kWaveGroups;           // vectors of a row
  __shared__ u32x4_t stage[4][16 * (kRow + 1)];  // a vector of padding per row
  const unsigned group_blocks = unsigned((a.G + kRestoreGroups - 1) / kRestoreGroups);
  const int wave = wave_index(), lane = threadIdx.x & 63;
  const int o0 = int(blockIdx.x / group_blocks) * 16;
  const int r = lane >> 2, w = lane & 3;
  const int g0 = int(blockIdx.x % group_blocks) * kRestoreGroups + wave * kWaveGroups;
  if (g0 >= a.G) return;
  const int o = min(o0 + r, a.O - 1);  // rows past O expand the last row, groups past G the last group: not stored
  RestoreWord in[kWaveGroups];
#pragma unroll
  for (int i = 0; i < kWaveGroups; ++i) in[i] = load_word(a, min(g0 + i, a.G - 1), o, w);
#pragma unroll
  for (int i = 0; i < kWaveGroups; ++i) {
    u32x4_t v[4];
    restore_word<WDT>(in[i], a.sdt, v);
#pragma unroll
    for (int b = 0; b < 4; ++b) stage[wave][r * (kRow + 1) + i * 16 + b * 4 + w] = v[b];  // vector 4 w + b of the group
  }
  wave_lds_order();
  const size_t K = size_t(a.G) * 128;
#pragma unroll
  for (int k = 0; k < 16 * kRow / 64; ++k) {
    const int unit = k * 64 + lane, row = unit / kRow, u = unit % kRow;
    const u32x4_t out = stage[wave][row * (kRow + 1) + (u & ~15) + (u & 3) * 4 + ((u >> 2) & 3)];
    if (o0 + row < a.O && g0 + (u >> 4) < a.G) {
      uint16_t* dst = a.weight + size_t(o0 + row) * K + size_t(g0) * 128 + u * 8;
      if (a.weight16) {
        *reinterpret_cast<u32x4_t*>(dst) = out;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[j] = uint16_t(out[j >> 1] >> (16 * (j & 1)));
      }
    }
  }
}

// With a column permutation.  A workgroup stages `rows_per_block` whole rows
// in LDS (rows_per_block * K * 2 bytes, zeroed first), scatters each expanded
// value to its permuted column there, and then writes the rows out in order
// with 16-byte stores, so a scattered permutation costs LDS scatter and not
// scattered HBM stores.  Entries outside [0, K) are skipped; a column no entry
// names stays zero.  A lane keeps the 32 entries of its word over the rows.
constexpr int kRestoreStageThreads = 512;

template <int WDT>
__global__ __launch_bounds__(kRestoreStageThreads) void w3_restore_permuted_kernel(RestoreArgs a, int rows_per_block) {
  extern __shared__ uint4 stage_vec[];
  uint16_t* stage = reinterpret_cast<uint16_t*>(stage_vec);
  const int K = a.G * 128;
  const int o0 = int(blockIdx.x) * rows_per_block;
  const int rows = min(rows_per_block, a.O - o0);
  const int vecs = rows * K / 8;
  for (int i = threadIdx.x; i < vecs; i += kRestoreStageThreads) stage_vec[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  // items (row slice, word): neighbouring lanes take the words of neighbouring groups
  const int words = a.G * 4;
  const int slices = max(1, min(rows, kRestoreStageThreads / words));
  for (int it = threadIdx.x; it < words * slices; it += kRestoreStageThreads) {
    const int word = it % words, slice = it / words;
    const int16_t* entries = a.perm + word * 32;
    unsigned cols[16];  // two entries each
    if (a.perm16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 p = reinterpret_cast<const uint4*>(entries)[j];
        cols[4 * j] = p.x, cols[4 * j + 1] = p.y, cols[4 * j + 2] = p.z, cols[4 * j + 3] = p.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j)
        cols[j] = unsigned(uint16_t(entries[2 * j])) | (unsigned(uint16_t(entries[2 * j + 1])) << 16);
    }
    for (int r = slice; r < rows; r += slices) {
      u32x4_t v[4];
      restore_word<WDT>(load_word(a, word >> 2, o0 + r, word & 3), a.sdt, v);
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const int col = int(int16_t(cols[j >> 1] >> (16 * (j & 1))));
        if (unsigned(col) < unsigned(K)) stage[r * K + col] = uint16_t(v[j >> 3][(j >> 1) & 3] >> (16 * (j & 1)));
      }
    }
  }
  __syncthreads();
  uint16_t* dst = a.weight + size_t(o0) * K;
  if (a.weight16) {
    uint4* dst_vec = reinterpret_cast<uint4*>(dst);
    for (int i = threadIdx.x; i < vecs; i += kRestoreStageThreads) dst_vec[i] = stage_vec[i];
  } else {
    for (int i = threadIdx.x; i < rows * K; i += kRestoreStageThreads) dst[i] = stage[i];
  }
}

bool launch_restore(int weight_dtype, const RestoreArgs& a, hipStream_t s) {
  const bool bf = weight_dtype == kBF16;
  if (!a.perm) {
    const size_t blocks = size_t((a.O + 15) / 16) * size_t((a.G + kRestoreGroups - 1) / kRestoreGroups);
    if (blocks > size_t(INT32_MAX)) return false;
    hipLaunchKernelGGL(bf ? w3_restore_kernel<kBF16> : w3_restore_kernel<kF16>, dim3(unsigned(blocks)), dim3(256), 0, s, a);
    return true;
  }
  const int K = a.G * 128, rows = kRestoreStageBytes / (2 * K) > 1 ? kRestoreStageBytes / (2 * K) : 1;
  hipLaunchKernelGGL(bf ? w3_restore_permuted_kernel<kBF16> : w3_restore_permuted_kernel<kF16>,
                     dim3(unsigned((a.O + rows - 1) / rows)), dim3(kRestoreStageThreads), size_t(rows) * K * 2, s, a, rows);
  return true;
}

}  // namespace fx
