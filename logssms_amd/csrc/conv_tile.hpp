// Tokens per block of conv_vec_kernel (conv.hip).
//
// A block walks its tile serially, about 0.6 us a token when alone on its CU,
// so a 32-token tile took 23-29 us at any T below 4096; a shorter tile
// re-reads the W-1 rows before it (from L2).  The tile is the shortest (in
// whole groups of 4, the window ring's period, or 2, and at most 32) with which
// all blocks run at once: `blocks_per_cu` of them on each of 256 CUs, shared
// among the slabs of 2048 channels.  Past that point the tile stays at 32 and
// the blocks run in rounds.  q/k pass, 2 slabs, us at tile 32 / 16 / 8 / 4 / 2:
// T 300: 23.8 / 13.5 / 9.0 / 6.7 / 5.8; 2048: 28.9 / 15.9 / 13.1 / 13.2 / 15.9;
// 8192: 36.8 / 30.3 / 30.8 / 35.8 / 45.0; 16384: 63.4 / 64.4 / 65.7 / 70.5 /
// 87.8.  A tile that leaves a few blocks to a second round costs what the longer
// one gains (8192 tokens, us, tile 24 / 28 / 32: front end of 3 slabs, 1026
// blocks of 24 tokens, 45.9 / 39.3 / 38.3; plain bf16 conv of 2 slabs, where 3
// blocks fit a CU, tile 16 / 24 / 32: 28.7 / 24.9 / 25.1).
#pragma once

#include <cstdint>

namespace gdn {

constexpr int kVTok = 32, kVTokMin = 2;

inline int conv_tile(int64_t tokens, int64_t slabs, int blocks_per_cu) {
  const int64_t blocks = 256 * blocks_per_cu / slabs;  // resident blocks of one slab
  const int64_t least = blocks > 0 ? (tokens + blocks - 1) / blocks : kVTok;
  if (least <= kVTokMin) return kVTokMin;
  return static_cast<int>(least >= kVTok ? kVTok : (least + 3) / 4 * 4);
}

}  // namespace gdn
