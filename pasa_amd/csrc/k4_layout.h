// LDS images shared by the K4 kernels (head_dim 128 and 64) and the pack kernel that writes
// their phase-2 operands.
#pragma once

#include "common.h"

namespace pasa {

constexpr int kGroup = 32;  // key blocks per group of the first-order correction

// V^ transposed (feature rows e of the group's 32 block sums), as the 16x16x32 MFMA reads
// it: rows of 80 bytes (64 + 16 of padding, so that the 16-byte reads of 16 consecutive
// rows hit 16 distinct chunk positions), and chunk c of a row holding blocks 4c .. 4c + 3
// and 16 + 4c .. 16 + 4c + 3: the 8 k-slots a lane of group c feeds to one MFMA, in the
// order its P-bar operand holds them.
constexpr int kVtRow = 80;
__host__ __device__ __forceinline__ constexpr int vt_block_of(int chunk, int i) {
  return ((i & 4) << 2) | (chunk << 2) | (i & 3);
}

// Tiles of D-feature rows, 16-byte chunk c of row r stored at c ^ kx(r) (K, kbar, Hbar^T: the
// reads of 16 rows at one chunk touch 16 distinct 16-byte bank groups) or c ^ vx(r) (V: the
// transposing reads of 8 rows x 2 chunks do).  At D = 64 two rows share a 256-byte bank line, so
// the swizzle takes the row's bits from the second on.  Both depend on r mod 16 only.
template <int D>
struct K4Tile {
  static_assert(D == 128 || D == 64, "head dims of the tuned kernels");
  static constexpr int ROWB = 2 * D;
  __host__ __device__ static constexpr int kx(int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); }
  __host__ __device__ static constexpr int vx(int r) { return D == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); }
  __host__ __device__ static constexpr int k_byte(int row, int col) {
    return row * ROWB + (((col >> 3) ^ kx(row)) << 4) + (col & 7) * 2;
  }
};

// Phase-2 pack image, split between the two LDS tile buffers: [Hbar^T: D rows in the K layout] ->
// K buffer; [kbar: 32 rows in the K layout][V^ transposed: D rows x kVtRow] -> V buffer.
// Both parts are whole multiples of 4 KB, so the four waves of a workgroup split their 1 KB
// direct loads evenly.
template <int D>
struct K4Pack {
  static constexpr int HT_BYTES = D * 2 * D;
  static constexpr int KB_OFF = 0;                       // within the V-buffer part
  static constexpr int VT_OFF = 32 * 2 * D;
  static constexpr int RAW2 = VT_OFF + D * kVtRow;
  static constexpr int PART2 = (RAW2 + 4095) / 4096 * 4096;
  static constexpr int BYTES = HT_BYTES + PART2;
  static_assert(HT_BYTES % 4096 == 0, "pack split");
};

}  // namespace pasa
