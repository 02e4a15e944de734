// Scratch memory of the device raster: which windows are rasterized by tiles, the
// room of the tiles' lists, and what is tried where they do not fit.  Shared by the
// launches and the host code that allocates (also compiled by the CPU tests, so it
// includes no HIP header).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace drvk {

constexpr int kTile = 16;
constexpr uint32_t kTileSpan = 64;  // triangles that touch more tiles go to the records that every tile looks through
constexpr uint32_t kHeadWords = 8;  // counters before those of the tiles

// Windows of at least this many tiles take the tiled raster: a tile is one
// workgroup's work, and a small window's few tiles hold many triangles each
// and leave the chip idle.  us in two passes / tiled, of 1.0M, 157k, 12k and 2176
// (large) triangles:
//   view 256x256 (256 tiles)   155 / 402   78 / 188   65 / 77    55 / 45
//   view 400x240 (375)         293 / 276  103 / 138   64 / 68    60 / 43
//   view 480x270 (510)         407 / 239  121 / 125   68 / 72    66 / 45
//   view 640x360 (920)         683 / 198  203 / 107  133 / 69   121 / 49
//   RSM 256x256                 89 / 411   71 / 172   63 / 94    98 / 72
//   RSM 512x512 (1024)         269 / 255  116 / 146   84 / 98   191 / 82
//   RSM 1024x1024             1633 / 266  380 / 187  198 / 136  423 / 129
constexpr int kMinTiles = 384;

inline int tile_count(int w, int h) { return ((w + kTile - 1) / kTile) * ((h + kTile - 1) / kTile); }
// Tile coordinates have 12 bits, and the pairs of 2^24 triangles count in 32.
inline bool tiled(int w, int h, uint32_t n_tri) {
  return tile_count(w, h) >= kMinTiles && w <= 65536 && h <= 65536 && n_tri <= (1u << 24);
}

// Room of the tiled raster's lists and records; what passes it is drawn by the
// two passes before the tiles.
struct TileRoom {
  uint32_t pairs, wide, cut;
  bool all;  // everything fits that could come: no triangle is left to the two passes
};
inline TileRoom tile_room(int w, int h, uint32_t n_tri) {
  constexpr uint64_t kWideLooks = 1u << 30;  // of all tiles at wide records: ~1 ms
  const uint64_t n = n_tri, tiles = static_cast<uint64_t>(tile_count(w, h));
  TileRoom r;
  r.pairs = static_cast<uint32_t>(std::min<uint64_t>(2 * kTileSpan * n, 4 * n + (1u << 22)));
  r.cut = static_cast<uint32_t>(std::min<uint64_t>(2 * n, 65536));
  r.wide = static_cast<uint32_t>(std::min<uint64_t>({2 * n, 65536, std::max<uint64_t>(256, kWideLooks / tiles)}));
  r.all = r.pairs == 2 * kTileSpan * n && r.wide == 2 * n && r.cut == 2 * n;
  return r;
}

// uint32 of the lists: the two passes' (the least that the launches do with) and
// the tiled raster's: records of four words, a counter and a start for each
// tile, clipped and left-out triangles, pairs of three words and their items.
inline size_t raster_least_words(uint32_t n_tri) { return static_cast<size_t>(n_tri) + 1; }
inline size_t raster_work_words(int w, int h, uint32_t n_tri) {
  if (!tiled(w, h, n_tri)) return raster_least_words(n_tri);
  const TileRoom room = tile_room(w, h, n_tri);
  return kHeadWords + 2 * static_cast<size_t>(n_tri) + 2 * static_cast<size_t>(tile_count(w, h)) +
         4 * (static_cast<size_t>(room.pairs) + room.wide + room.cut);
}

// Reserves `words`, or `least` where those do not fit.  reserve(n) returns 0,
// no_memory or another error.  refused: the least number that did not fit so
// far, not tried again.
template <typename Reserve>
int reserve_raster_words(size_t words, size_t least, size_t* refused, int no_memory, Reserve&& reserve) {
  if (words < *refused || words == least) {
    const int rc = reserve(words);
    if (rc != no_memory || words == least) return rc;
    *refused = words;
  }
  return reserve(least);
}

}  // namespace drvk
