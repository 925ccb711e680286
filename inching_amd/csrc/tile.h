// Shapes of the tile form of the matrix-free product, shared by its construction and its kernel.
#pragma once
#include <cstdint>

// tile atoms x lanes per atom: a workgroup's threads, one tile. The kernel is instantiated
// for these shapes alone.
inline bool inch_tile_shape_ok(int32_t tile, int32_t lanes) {
  return (tile == 64 && lanes == 8) || (tile == 32 && lanes == 16) || (tile == 16 && lanes == 32);
}

// Records of a tile's union: with one dummy record per atom they fit 64 KiB of LDS, so that a
// record's byte offset fits the 16 bits of a pair entry.
inline int32_t inch_tile_max_union(int32_t tile) { return 65536 / 48 - tile; }
