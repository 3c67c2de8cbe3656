// What the 16-bit prefill kernels (prefill.hip, prefill_rows.hip) share: the
// K/V tile geometry in LDS.
#pragma once

#include "common.h"

namespace ca {

// K/V tiles in LDS: rows of 2 D bytes, unpadded, the 16-byte chunk c of row r
// at position c ^ swz(r) (see prefill.hip).
template <int D>
struct PfGeom {
  static_assert(D == 64 || D == 128, "head dim");
  static constexpr int kBN = 64;                     // keys per tile
  static constexpr int kRowB = D * 2;                // bytes per K/V row
  static constexpr int kLpr = kRowB / 16;            // 16-byte chunks per row
  static constexpr int kRpk = 1024 / kRowB;          // rows per 1-KB load
  static constexpr int kTileB = kBN * kRowB;         // bytes per K (or V) tile
  static constexpr int kStageB = 2 * kTileB;         // K tile then V tile
  static constexpr int kNKS = D / 16;                // QK k-steps
  static constexpr int kNOB = D / 32;                // O^T row blocks
  __device__ static __forceinline__ int swz(int r) {
    return D == 128 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
  }
};

}  // namespace ca
