// The W3 GEMM's activation packing and K-split finish (the product: w3_gemm.h).
#include "common.h"
#include "w3_gemm_launch.h"

namespace fx {

// Unit of (row, 8-column unit c of the payload's order): batch c / 64, k-block
// c % 64 / 16, step c % 16, at [row block][batch][step][tile][k-block][row % 16].
__device__ __forceinline__ size_t packed_unit(int row, int c, int mt, int batches) {
  const int block = row / (16 * mt), tile = (row >> 4) - block * mt;
  return (((size_t(block) * batches + (c >> 6)) * 16 + (c & 15)) * mt + tile) * 64 + ((c >> 4) & 3) * 16 + (row & 15);
}

// Identity order: a thread copies the four units of one word of one row (64
// contiguous bytes); rows past M and columns past K become zeros.  A wave covers
// 16 rows x 4 k-blocks, so it stores whole operands.
__global__ __launch_bounds__(256) void gemm_pack_kernel(GemmPackArgs a) {
  const int batches = (a.K + 511) / 512;
  const int wave = int(blockIdx.x) * 4 + int(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int w = wave & 3, batch = (wave >> 2) % batches, tile = (wave >> 2) / batches;
  const int row = tile * 16 + (lane & 15), c0 = batch * 64 + (lane >> 4) * 16 + 4 * w;
  if (tile >= (a.M + 16 * a.mt - 1) / (16 * a.mt) * a.mt) return;
  const bool real = row < a.M && c0 * 8 < a.K;  // a k-block is one group: all or none of it
  const uint4* src = reinterpret_cast<const uint4*>(a.x + size_t(row) * a.K + c0 * 8);
  uint4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = real ? src[i] : make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) a.packed[packed_unit(row, c0 + i, a.mt, batches)] = v[i];
}

// With a column permutation: a workgroup copies R rows into LDS and gathers its share
// of the columns from there (random 2-byte reads of HBM would cost a cache line each).
// Entries outside [0, K) read zero.
constexpr int kPackThreads = 512;
template <int R>
__global__ __launch_bounds__(kPackThreads) void gemm_pack_permuted_kernel(GemmPackArgs a) {
  extern __shared__ uint4 pack_rows[];
  const int batches = (a.K + 511) / 512, row0 = int(blockIdx.x) * R, vecs = a.K / 8;
  const int cols = batches * 64, per = (cols + int(gridDim.y) - 1) / int(gridDim.y);  // 8-column units, units a share
  const int c0 = int(blockIdx.y) * per, c1 = min(cols, c0 + per);
  const int rr = int(threadIdx.x) % R, cstep = kPackThreads / R;
  int c = c0 + int(threadIdx.x) / R;  // neighbouring lanes: rows of one unit, contiguous in the output
  const uint4 zero = make_uint4(0, 0, 0, 0);
  const uint4* perm = reinterpret_cast<const uint4*>(a.perm);
  uint4 p = c < c1 && c < vecs ? perm[c] : zero;  // in flight over the copy
  const uint4* src = reinterpret_cast<const uint4*>(a.x) + size_t(row0) * vecs;
#pragma unroll
  for (int k = 0; k < R; ++k)
    for (int i = threadIdx.x; i < vecs; i += kPackThreads) pack_rows[k * vecs + i] = row0 + k < a.M ? src[k * vecs + i] : zero;
  __syncthreads();
  const uint16_t* row = reinterpret_cast<const uint16_t*>(pack_rows + rr * vecs);
  uint4* dst = a.packed + packed_unit(row0, 0, a.mt, batches) + rr;
  while (c < c1) {
    const int next = c + cstep;
    const uint4 pn = next < c1 && next < vecs ? perm[next] : zero;
    uint4 v = zero;
    if (c < vecs) {
      const unsigned pw[4] = {p.x, p.y, p.z, p.w};
      unsigned o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int lo = int(int16_t(pw[i])), hi = int(pw[i]) >> 16;
        const unsigned a0 = unsigned(lo) < unsigned(a.K) ? row[lo] : 0u;
        const unsigned a1 = unsigned(hi) < unsigned(a.K) ? row[hi] : 0u;
        o[i] = a0 | (a1 << 16);
      }
      v = make_uint4(o[0], o[1], o[2], o[3]);
    }
    dst[size_t(((c >> 6) * 16 + (c & 15)) * a.mt) * 64 + ((c >> 4) & 3) * 16] = v;
    c = next;
    p = pn;
  }
}

// Rows a workgroup stages: four write 64 contiguous bytes of the output together;
// few rows run one to a workgroup, shared over more of them, since their copy and
// gather are then the latency (37 rows of 4096: 4.8 us with four, see the kernel trace).
void launch_gemm_pack(const GemmPackArgs& a, hipStream_t s) {
  const int batches = (a.K + 511) / 512, tiles = (a.M + 16 * a.mt - 1) / (16 * a.mt) * a.mt, rows = tiles * 16;
  if (!a.perm) {
    hipLaunchKernelGGL(gemm_pack_kernel, dim3(unsigned(tiles * batches)), dim3(256), 0, s, a);
    return;
  }
  const int want = rows <= 64 ? 1 : rows <= 128 ? 2 : 4, fits = 65536 / (2 * a.K);  // at most 64 KB of LDS
  const int r = want == 4 && fits >= 4 ? 4 : want >= 2 && fits >= 2 ? 2 : 1;
  const unsigned blocks = unsigned(rows / r), share = blocks < 128 ? 4 : blocks < 256 ? 2 : 1;
  const auto kernel = r == 4 ? gemm_pack_permuted_kernel<4> : r == 2 ? gemm_pack_permuted_kernel<2>
                                                                   : gemm_pack_permuted_kernel<1>;
  hipLaunchKernelGGL(kernel, dim3(blocks, share), dim3(kPackThreads), size_t(r) * a.K * 2, s, a);
}

// out = the splits' partials in split order, plus the bias, rounded once; four
// outputs per thread.
template <int XDT>
__global__ __launch_bounds__(256) void gemm_finish_kernel(GemmArgs a, int splits) {
  const size_t total = size_t(a.M) * a.O, at = (size_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (at >= total) return;
  if (a.vec) {
    float4 sum = *reinterpret_cast<const float4*>(a.partial + at);
    for (int k = 1; k < splits; ++k) {
      const float4 p = *reinterpret_cast<const float4*>(a.partial + size_t(k) * total + at);
      sum.x += p.x, sum.y += p.y, sum.z += p.z, sum.w += p.w;
    }
    if (a.bias) {
      const int o = int(at % unsigned(a.O));
      sum.x += to_f32<XDT>(a.bias[o]), sum.y += to_f32<XDT>(a.bias[o + 1]);
      sum.z += to_f32<XDT>(a.bias[o + 2]), sum.w += to_f32<XDT>(a.bias[o + 3]);
    }
    *reinterpret_cast<uint2*>(a.out + at) =
        uint2{unsigned(from_f32<XDT>(sum.x)) | (unsigned(from_f32<XDT>(sum.y)) << 16),
              unsigned(from_f32<XDT>(sum.z)) | (unsigned(from_f32<XDT>(sum.w)) << 16)};
    return;
  }
  for (size_t i = at; i < at + 4 && i < total; ++i) {
    float sum = a.partial[i];
    for (int k = 1; k < splits; ++k) sum += a.partial[size_t(k) * total + i];
    if (a.bias) sum += to_f32<XDT>(a.bias[i % unsigned(a.O)]);
    a.out[i] = from_f32<XDT>(sum);
  }
}

void launch_gemm_finish(int xdt, const GemmArgs& a, int splits, hipStream_t s) {
  const dim3 grid(unsigned((size_t(a.M) * a.O + 1023) / 1024)), block(256);
  if (xdt == kBF16)
    hipLaunchKernelGGL(gemm_finish_kernel<kBF16>, grid, block, 0, s, a, splits);
  else
    hipLaunchKernelGGL(gemm_finish_kernel<kF16>, grid, block, 0, s, a, splits);
}

}  // namespace fx
