// Host-side declarations of the split-contract GEMV (w3_split.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fx {

struct SplitArgs {
  const uint16_t* x;
  const uint8_t* planes;
  const uint16_t* scales;
  const uint8_t* zeros;  // null: zero-point 4
  const int16_t* perm;   // null: the identity
  float* partial;        // [splits, O], or null (one split: only out is written)
  uint16_t* out;         // [O], or null (only the partials are written)
  int O, G;
  int gps;      // groups per split
  int sdt;      // scale dtype
  int decoded;  // weights with |q - z| = 3 rounded to bf16
  int x16, perm16;  // 16-byte aligned
  int slot_shift;   // log2 of the groups of a batch in one split (launch_split sets it)
};

constexpr int kSplitMaxColumns = 16384;

// The K splits that the kernel forms: whole four-group batches, or one or two groups.
inline bool split_kernel_takes(int G, int gps) {
  return G * 128 <= kSplitMaxColumns && (gps >= G || gps % 4 == 0 || gps == 1 || gps == 2);
}
void launch_split(int xdt, SplitArgs a, hipStream_t s);

}  // namespace fx
