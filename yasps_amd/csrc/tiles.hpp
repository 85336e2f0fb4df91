// Tiled symmetric operator of the PCG product.
//
// The mirrored full block-CSR reads every off-diagonal block twice. Here the block rows
// are cut into tiles of kTileRows rows that lie close together in space; a block whose two
// rows share a tile is stored once and serves both (y_r += B x_c in registers,
// y_c += B^T x_r in the tile's LDS), a block between two tiles is stored in both. One
// thread owns one row of the tile (two threads with kTileTpr = 2) and walks its entries,
// which lie in slices of 64 rows: entry j of the slice's lane l at slice_start + 64 j + l,
// so the lanes of a wavefront read 64 consecutive values of each component.
#pragma once
#include "common.hpp"

namespace ysp {

constexpr uint32_t kTileRows = YSP_TILE_ROWS;
constexpr uint32_t kTileCut = 1u << 31;       // entry word: the column lies in another tile
constexpr uint32_t kTileNoSource = 0xffffffffu;
constexpr uint32_t kTileMaxRow = 96;          // longest row (entries) a tile takes

struct TiledView {
  const uint32_t* rows;         // [nv] block row at every tile position
  const uint32_t* lens;         // [nv] entries of the row at that position
  const uint32_t* slice_start;  // [slices + 1] first entry of each slice of 64 positions
  const uint32_t* entry;        // [entries] the column's position: in the tile, or
                                // kTileCut | its position in the operator
  uint32_t entries;             // including the slices' padding (read by nothing; without it the
                                // product kernel is scheduled worse: a 64^3-cell cube's solve
                                // 10.24 -> 10.30 ms)
};

template <typename VT>
struct Tiled {
  TiledView t;
  const VT* v;                  // component i of entry k at tile_value(k) + 64 i
};

// The nine values of 64 consecutive entries lie together, component by component: a wavefront
// reads 64 entries as one run of 4,608 bytes at fixed offsets from one address.
__host__ __device__ __forceinline__ size_t tile_value(uint32_t k) {
  return static_cast<size_t>(k / 64) * 576 + k % 64;
}

}  // namespace ysp
