// Host-side declarations of the W3 dequantize (w3_restore.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fx {

struct RestoreArgs {
  const uint8_t* planes;
  const uint16_t* scales;
  const uint8_t* zeros;  // null: zero-point 4
  const int16_t* perm;   // null: the identity
  uint16_t* weight;      // [O, 128 G]
  int O, G;
  int sdt;       // scale dtype
  int weight16;  // weight 16-byte aligned
  int perm16;    // perm 16-byte aligned
};

constexpr int kRestoreGroups = 8;           // identity order: groups per workgroup
constexpr int kRestoreStageBytes = 65536;  // permuted: rows per workgroup = max(1, this / 2K)

// False when the grid would exceed its limit.
bool launch_restore(int weight_dtype, const RestoreArgs& a, hipStream_t s);

}  // namespace fx
