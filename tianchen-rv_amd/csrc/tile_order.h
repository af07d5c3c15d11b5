// tile_order.h -- work-group order of the plain-row and repack GEMMs (gemm_batch.hip,
// gemm_rows16.hip, gemm_repack.hip) over the 8 XCDs.
//
// The hardware deals work-groups to the XCDs in turn, x fastest, so in a grid of (8, y, z)
// blockIdx.x is the XCD.  Each XCD takes a run of consecutive tiles, token tiles fastest (the
// tiles of a row tile read the same weights through one L2).  The runs are of whole row tiles
// while the longest fits one work-group a CU (2 x 113 x 256 Q4_0 2.6 us, 2.9 over all XCDs); past
// that they differ by one tile at most: whole row tiles put twice a round on some XCDs at
// 35 x 7 tiles (2220 x 219 x 2304 Q8_0 16.6 -> 19.9 us) and all of one row tile on one.
#pragma once

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define TCRV_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define TCRV_HOST_DEVICE inline
#endif

namespace tcrv {

constexpr uint32_t kXcds = 8, kXcdCus = 32;
// Slots of an XCD past this many go on in z (the last z is part empty).
constexpr uint32_t kSlotsY = 512;
// A launch takes fewer tiles than this (z is 65535 at most).
constexpr size_t kMaxTiles = static_cast<size_t>(kXcds) * kSlotsY * 65535;

// The order of a launch.  The kernels take units and inv as their first arguments and count the
// tiles from their own: what a wave needs before its first loads stays within the 14
// argument dwords that the command processor preloads (an argument past them, or a read of
// gridDim, is a scalar load that the loads wait for: 0.1-0.4 us of a 3-10 us kernel).
struct TileOrder {
  uint32_t units;             // what the runs are counted in: row tiles or tiles
  uint32_t inv;               // 2^32 / token tiles, rounded down (2^32 - 1 for one)
  uint32_t slots_y, slots_z;  // the grid's y and z
};

struct TilePos {
  uint32_t tm, tn;
  bool live;
};

// False for kMaxTiles tiles and more.
inline bool tile_order(size_t row_tiles, size_t tok_tiles, TileOrder *o) {
  if (row_tiles >= kMaxTiles || tok_tiles >= kMaxTiles || row_tiles * tok_tiles >= kMaxTiles)
    return false;
  const uint32_t rows = static_cast<uint32_t>(row_tiles), toks = static_cast<uint32_t>(tok_tiles);
  const uint32_t each = (rows + kXcds - 1) / kXcds;  // row tiles of the longest run
  const bool by_row = each <= kXcdCus / toks;
  o->units = by_row ? rows : rows * toks;
  o->inv = toks == 1 ? 0xffffffffu : static_cast<uint32_t>((1ull << 32) / toks);
  const uint32_t slots = by_row ? each * toks : (o->units + kXcds - 1) / kXcds;
  o->slots_y = slots < kSlotsY ? slots : kSlotsY;
  o->slots_z = (slots + kSlotsY - 1) / kSlotsY;
  return true;
}

// The tile of work-group (x, y, z): XCD x's run is units x / 8 .. units (x + 1) / 8 - 1.
TCRV_HOST_DEVICE TilePos xcd_tile(uint32_t units, uint32_t row_tiles, uint32_t tok_tiles,
                                  uint32_t inv, uint32_t x, uint32_t y, uint32_t z) {
  const uint32_t unit = units == row_tiles ? tok_tiles : 1;
  const uint32_t tile = units * x / kXcds * unit + y + kSlotsY * z;
  // tile / tok_tiles: the product with inv falls short by one at most, which the sign of the
  // rest tells (a comparison here leaves the scalar registers, and the addresses with it:
  // 0.2-0.6 us)
  const uint32_t q = static_cast<uint32_t>((static_cast<uint64_t>(tile) * inv) >> 32);
  const uint32_t r = tile - q * tok_tiles, up = (tok_tiles - 1 - r) >> 31;
  TilePos p;
  p.live = tile < (units * x + units) / kXcds * unit;
  p.tm = q + up;
  p.tn = r - up * tok_tiles;
  return p;
}

}  // namespace tcrv
