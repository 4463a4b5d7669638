// Selection lists of the union attention passes (sparse_attn_union.hip): for every block of 16
// queries and every tile of 256 keys, the keys that at least one query of the block selected,
// with each key's 16-bit query set, laid out for the matrix-core operands of a wave.
#pragma once

#include "gw_dense.h"

namespace gw {

constexpr int kUQ = 16;                // rows (queries) per block
constexpr int kUTile = 256;            // columns (keys) per tile
constexpr int kURec = 1024;            // bytes of one (block, tile) record
constexpr int kUTileBytes = 65536;     // one head's K and V rows of a tile
constexpr int kUPlane = 16384;         // one 32-dim half of K or V of a tile

// A (block, tile) record. The tile's selected keys fill slots in an order that spreads
// consecutive slots over the key's residues mod 8 (conflict-free LDS rows, see
// union_tiles_kernel); steps of 32 slots, two groups of 4 steps.
//   bytes 256 g + 4 l, lane l of a wave: bit 8 j + 7 - 2 s - f is clear when query l % 16
//     selected the key of slot 32 (4 g + s) + 16 f + 4 (l / 16) + j (s, j < 4, f < 2).
//   bytes 512 + 256 g + 64 s + 4 i: the LDS row offsets (union_row) of slots 32 (4 g + s) + i
//     (low half) and + 16 + i (high half); unused slots hold row 0 and no query.
//     The first of them also holds the units in use, slots / 16 rounded up (0..16), in the low
//     four bits of its low half (units % 16) and of its high half (units / 16). The second
//     group (g = 1) is written only when units > 8.

// LDS offset of a tile row inside a plane: 64-byte rows, with bits 4-5 set to the row's swizzle,
// so that the 16-byte chunk c of the row's 4 sits at union_row(r) ^ (c << 4).
__host__ __device__ __forceinline__ uint32_t union_row(uint32_t r) { return (r << 6) | (((r >> 1) & 3u) << 4); }

struct UnionListSizes {
  int ntiles;     // 256-key tiles
  int64_t nblk;   // 16-query blocks, padded to a multiple of kUMaxWaves
};
constexpr int kUMaxWaves = 16;
inline UnionListSizes union_list_sizes(int64_t T, int64_t S) {
  UnionListSizes u;
  u.ntiles = (int)((S + kUTile - 1) / kUTile);
  u.nblk = (T + kUQ * kUMaxWaves - 1) / (kUQ * kUMaxWaves) * kUMaxWaves;
  return u;
}

}  // namespace gw
