// The gather's inputs rendered on the device: a depth-tested triangle raster
// with the G-buffer fill (shader/fillgbuffer.frag) and the RSM fill and
// mip chain (shader/fillrsm.frag:24-62, shader/downsamplersm.frag:15-33,
// driven by rendering/renderer.cpp:1300-1339).
//
// Raster rules (the same as the host producer in csrc/inputs, which the
// tests compare against): triangles are projected and clipped against the
// near plane in FP64, pixel centres are sampled, both windings are accepted,
// a fragment with reverse-Z depth z in (0, 1] is kept, and of all fragments
// of a pixel the one with the largest depth wins, the lowest triangle index
// among equal depths.  Small windows (most RSMs) take a two-pass visibility
// buffer: pass 1 takes the 64-bit atomic max of the depth bits (non-negative
// doubles order like their bit patterns), pass 2 the atomic min of the index
// among the fragments that reached that depth.  Larger ones are rasterized tile
// by tile in registers.  A resolve pass then shades each pixel from its
// winning triangle.
#include <algorithm>

#include "drv_internal.hpp"
#include "k_common.hpp"
#include "raster_room.hpp"

namespace drvk {
namespace {

constexpr float kPiF = 3.14159265358979f;   // shader/utils.glsl:1
constexpr float kPi2F = 6.28318530717958f;  // shader/utils.glsl:2

struct ScreenTri {
  double x[3], y[3], z[3];
};

// Projection and near-plane clip (w - z >= 0 for the reverse-Z projection);
// returns the number of screen triangles (0..2).
__device__ int project_clip(const float* p, const double* vp, int w, int h, ScreenTri* out) {
  double clip[3][4];
  for (int v = 0; v < 3; ++v)
    for (int r = 0; r < 4; ++r)
      clip[v][r] = vp[4 * r + 0] * p[3 * v + 0] + vp[4 * r + 1] * p[3 * v + 1] + vp[4 * r + 2] * p[3 * v + 2] +
                   vp[4 * r + 3];
  double poly[4][4];
  int n = 0;
  for (int v = 0; v < 3; ++v) {
    const double* a = clip[v];
    const double* b = clip[(v + 1) % 3];
    const double da = a[3] - a[2], db = b[3] - b[2];
    if (da >= 0) {
      for (int k = 0; k < 4; ++k) poly[n][k] = a[k];
      ++n;
    }
    if ((da >= 0) != (db >= 0)) {
      const double t = da / (da - db);
      for (int k = 0; k < 4; ++k) poly[n][k] = a[k] + (b[k] - a[k]) * t;
      ++n;
    }
  }
  if (n < 3) return 0;
  double sx[4], sy[4], sz[4];
  for (int i = 0; i < n; ++i) {
    if (poly[i][3] <= 1e-12) return 0;
    sx[i] = (poly[i][0] / poly[i][3] * 0.5 + 0.5) * w;
    sy[i] = (poly[i][1] / poly[i][3] * 0.5 + 0.5) * h;
    sz[i] = poly[i][2] / poly[i][3];
  }
  int m = 0;
  for (int i = 1; i + 1 < n; ++i) {
    const int idx[3] = {0, i, i + 1};
    for (int k = 0; k < 3; ++k) {
      out[m].x[k] = sx[idx[k]];
      out[m].y[k] = sy[idx[k]];
      out[m].z[k] = sz[idx[k]];
    }
    ++m;
  }
  return m;
}

struct RasterArgs {
  const float* positions;  // [n_tri][9]
  uint32_t n_tri;
  double vp[16];
  int w, h;
  unsigned long long* zbits;  // [h][w] depth bits (0 = empty)
  uint32_t* tri;              // [h][w] winning triangle (0xffffffff = none)
  uint32_t* big;              // triangles whose screen box exceeds kBigPixels
  uint32_t* n_big;
};

// Triangles of a larger pixel box than this are listed and rasterized by a
// wave each (a thread's loop over them holds up the other 63), above the second
// bound by the workgroup.  256x256, 1.0M triangles of 3 box pixels: both passes
// 174 us at 512 with a workgroup for each listed triangle, 54 us at 24 (8: 107,
// 64: 59); nearly all of what is left is reading and projecting.
constexpr uint32_t kBigPixels = 24;
constexpr uint32_t kHugePixels = 4096;

// Screen-space setup of one clipped triangle piece: pixel box and edge data.
struct Setup {
  ScreenTri q;
  int px0, py0, bw, bh;
  double inv;
  bool ok;
};

__device__ __forceinline__ Setup setup_piece(const ScreenTri& q, int w, int h) {
  Setup st;
  st.q = q;
  st.ok = false;
  const double miny = fmin(fmin(q.y[0], q.y[1]), q.y[2]), maxy = fmax(fmax(q.y[0], q.y[1]), q.y[2]);
  const double minx = fmin(fmin(q.x[0], q.x[1]), q.x[2]), maxx = fmax(fmax(q.x[0], q.x[1]), q.x[2]);
  // Bounds in double first so that off-screen triangles cannot overflow int.
  const double fy0 = fmax(0.0, ceil(miny - 0.5)), fy1 = fmin(static_cast<double>(h - 1), floor(maxy - 0.5));
  const double fx0 = fmax(0.0, ceil(minx - 0.5)), fx1 = fmin(static_cast<double>(w - 1), floor(maxx - 0.5));
  if (!(fy0 <= fy1) || !(fx0 <= fx1)) return st;
  const double area = (q.x[1] - q.x[0]) * (q.y[2] - q.y[0]) - (q.x[2] - q.x[0]) * (q.y[1] - q.y[0]);
  if (area == 0.0) return st;
  st.inv = 1.0 / area;
  st.px0 = static_cast<int>(fx0);
  st.py0 = static_cast<int>(fy0);
  st.bw = static_cast<int>(fx1) - st.px0 + 1;
  st.bh = static_cast<int>(fy1) - st.py0 + 1;
  st.ok = true;
  return st;
}

// Visits pixels start, start + step, ... of the piece's box (row-major) and
// calls f(pixel index, depth) for every kept fragment.
template <typename F>
__device__ __forceinline__ void raster_piece(const Setup& st, int w, uint32_t start, uint32_t step, F&& f) {
  const ScreenTri& q = st.q;
  const int rows = static_cast<int>(step / static_cast<uint32_t>(st.bw)), cols = static_cast<int>(step % static_cast<uint32_t>(st.bw));
  int px = st.px0 + static_cast<int>(start % static_cast<uint32_t>(st.bw));
  int py = st.py0 + static_cast<int>(start / static_cast<uint32_t>(st.bw));
  const int end_x = st.px0 + st.bw, end_y = st.py0 + st.bh;
  for (; py < end_y; px += cols, py += rows + (px >= end_x ? 1 : 0), px -= px >= end_x ? st.bw : 0) {
    const double cy = py + 0.5, cx = px + 0.5;
    const double e0 = ((q.x[2] - q.x[1]) * (cy - q.y[1]) - (q.y[2] - q.y[1]) * (cx - q.x[1])) * st.inv;
    const double e1 = ((q.x[0] - q.x[2]) * (cy - q.y[2]) - (q.y[0] - q.y[2]) * (cx - q.x[2])) * st.inv;
    const double e2 = 1.0 - e0 - e1;
    if (e0 < 0 || e1 < 0 || e2 < 0) continue;
    const double z = e0 * q.z[0] + e1 * q.z[1] + e2 * q.z[2];
    if (!(z > 0.0) || z > 1.0) continue;  // a fragment must beat the cleared depth 0
    f(static_cast<size_t>(py) * w + px, z);
  }
}

// The screen triangle of a triangle wholly in front of the near plane (the
// operations project_clip performs for it).  Returns the vertices in front.
__device__ __forceinline__ int project_front(const float* p, const double* vp, int w, int h, ScreenTri& out,
                                             bool& degenerate) {
  int front = 0;
  degenerate = false;
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    double c[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      c[r] = vp[4 * r + 0] * p[3 * v + 0] + vp[4 * r + 1] * p[3 * v + 1] + vp[4 * r + 2] * p[3 * v + 2] +
             vp[4 * r + 3];
    front += c[3] - c[2] >= 0 ? 1 : 0;
    degenerate = degenerate || c[3] <= 1e-12;
    out.x[v] = (c[0] / c[3] * 0.5 + 0.5) * w;
    out.y[v] = (c[1] / c[3] * 0.5 + 0.5) * h;
    out.z[v] = c[2] / c[3];
  }
  return front;
}

// Small triangles: one thread each.  Large ones and those that reach behind
// the near plane are listed (first pass) or skipped (second pass) for the
// workgroup kernel, which clips them.
template <typename F>
__device__ __forceinline__ void raster_small(const RasterArgs& a, uint32_t t, bool list_big, F&& f) {
  float p[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) p[i] = a.positions[9 * static_cast<size_t>(t) + i];
  ScreenTri sc;
  bool degenerate;
  const int front = project_front(p, a.vp, a.w, a.h, sc, degenerate);
  if (front == 0) return;
  bool list = front < 3;
  if (!list && degenerate) return;
  Setup st;
  st.ok = false;
  if (!list) {
    st = setup_piece(sc, a.w, a.h);
    list = st.ok && static_cast<uint32_t>(st.bw) * static_cast<uint32_t>(st.bh) > kBigPixels;
  }
  if (list) {
    if (list_big) a.big[atomicAdd(a.n_big, 1u)] = t;
    return;
  }
  if (st.ok) raster_piece(st, a.w, 0u, 1u, f);
}

// Large triangles: a wave each, the huge ones among them the workgroup.
template <typename F>
__device__ __forceinline__ void raster_big(const RasterArgs& a, F&& f) {
  __shared__ uint32_t huge[4];
  const uint32_t n = *a.n_big, lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  for (uint32_t i0 = 4u * blockIdx.x; i0 < n; i0 += 4u * gridDim.x) {
    const uint32_t i = i0 + w;
    uint32_t later = 0u;  // pieces
    if (i < n) {
      const uint32_t t = a.big[i];
      ScreenTri sc[2];
      const int m = project_clip(a.positions + 9 * static_cast<size_t>(t), a.vp, a.w, a.h, sc);
      for (int s = 0; s < m; ++s) {
        const Setup st = setup_piece(sc[s], a.w, a.h);
        if (!st.ok) continue;
        if (static_cast<uint64_t>(st.bw) * static_cast<uint64_t>(st.bh) > kHugePixels)
          later |= 1u << s;
        else
          raster_piece(st, a.w, lane, 64u, [&](size_t px, double z) { f(t, px, z); });
      }
    }
    if (lane == 0u) huge[w] = later;
    __syncthreads();
    for (uint32_t k = 0; k < 4u; ++k) {
      const uint32_t pieces = huge[k];
      if (pieces == 0u) continue;
      const uint32_t t = a.big[i0 + k];
      ScreenTri sc[2];
      const int m = project_clip(a.positions + 9 * static_cast<size_t>(t), a.vp, a.w, a.h, sc);
      for (int s = 0; s < m; ++s) {
        if (!(pieces >> s & 1u)) continue;
        const Setup st = setup_piece(sc[s], a.w, a.h);
        raster_piece(st, a.w, threadIdx.x, 256u, [&](size_t px, double z) { f(t, px, z); });
      }
    }
    __syncthreads();
  }
}

// Empty pixels and no listed triangle, in one launch instead of three fills
// (15 us before a 256^2 RSM, 5 now).
__global__ __launch_bounds__(256) void k_raster_clear(RasterArgs a) {
  const size_t n = static_cast<size_t>(a.w) * a.h;
  const size_t first = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (size_t i = first; i < n; i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    a.zbits[i] = 0ull;
    a.tri[i] = 0xffffffffu;
  }
  if (first == 0) *a.n_big = 0u;
}

__global__ __launch_bounds__(256) void k_raster_depth(RasterArgs a) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.n_tri) return;
  raster_small(a, t, true, [&](size_t i, double z) {
    atomicMax(&a.zbits[i], static_cast<unsigned long long>(__double_as_longlong(z)));
  });
}

__global__ __launch_bounds__(256) void k_raster_depth_big(RasterArgs a) {
  raster_big(a, [&](uint32_t, size_t i, double z) {
    atomicMax(&a.zbits[i], static_cast<unsigned long long>(__double_as_longlong(z)));
  });
}

__global__ __launch_bounds__(256) void k_raster_id(RasterArgs a) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.n_tri) return;
  raster_small(a, t, false, [&](size_t i, double z) {
    if (static_cast<unsigned long long>(__double_as_longlong(z)) == a.zbits[i]) atomicMin(&a.tri[i], t);
  });
}

__global__ __launch_bounds__(256) void k_raster_id_big(RasterArgs a) {
  raster_big(a, [&](uint32_t t, size_t i, double z) {
    if (static_cast<unsigned long long>(__double_as_longlong(z)) == a.zbits[i]) atomicMin(&a.tri[i], t);
  });
}

// ---- the tiled raster ----------------------------------------------------
//
// For windows of many tiles.  Triangles are binned to the 16x16-pixel tiles
// their pixel boxes touch (count, start, fill); then one workgroup per tile
// keeps the tile's pixels in registers, one pixel per lane (a wave owns 8x8),
// and walks the tile's triangles, 256 at a time: every thread sets up one
// triangle in LDS, then every wave tests those that may touch it.  A pixel
// keeps the greatest FP64 depth and the lowest index at it, as the two passes
// above find with atomics.  The triangle's thread settles for each wave by FP32
// planes with an error margin whether all its pixels are outside or behind, the
// wave then for its lanes; the FP64 test, with the operations of raster_piece,
// runs when a lane is left.
//
// Triangles of more than kTileSpan tiles are records that every tile looks
// through and gathers to whole batches.  Lists and records have fixed room
// (tile_room): what finds none is drawn by the two passes above before the tiles,
// whose pixels then start from that, so a scene past the room costs no more than
// the two passes.  1920x1080 / 3840x2160, two passes for all of it and this:
// 200000 triangles of some 50 tiles (twice the room) 5.4 / 5.4 and 0.32 / 0.62 ms,
// 1.0M of some 30 (four times) 23 / 23 and 1.4 / 1.9, 30000 of 1000 tiles 8.2 / 8.6
// and 0.89 / 2.8.  (With 4 n + 2^16 pairs and all others as records that each tile
// took in batches of 256, hits or not: 8.5 / 15.9, 23 / 53 and 4.4 / 12.9 ms.)
//
// 1920x1080, 1.0M triangles in 2000 boxes (74M box pixels, 18 layers deep):
// the two passes 1660 us, of it atomics and FP64 tests of hidden fragments;
// count 48, near-plane pieces 11, starts 5, fill 8, tiles 119 us: 48 000 vector
// instructions on each SIMD, those in FP64 of four cycles or more, in 286 000
// cycles, with the waves waiting half of their time.

constexpr int kTileGroups = 16;     // tiles of which a wave adds up the pairs before its atomics

struct TileRecord {
  uint32_t x, y;  // first | last << 16 tile
  uint32_t tri;
  uint32_t piece;  // 0, 1: piece of a triangle cut by the near plane; 2: not cut
};
constexpr uint32_t kRecordItem = 0x80000000u;  // an item of a tile's list: a triangle, or this and a record

struct TilePair {
  uint32_t item, tile, rank;  // rank: place in the tile's list
};
constexpr uint32_t kNoTile = 0xffffffffu;

struct TileArgs {
  RasterArgs r;         // r.big: triangles that found no room
  int tiles_x, tiles_y;
  uint32_t capacity;    // pairs
  uint32_t wide_capacity, cut_capacity;  // records
  uint32_t* head;       // {wide records, clipped triangles, pairs, records in lists, r.n_big, room taken by lists, 0, 0}, then the counts
  uint32_t* count;      // [tiles]
  uint32_t* start;      // [tiles]
  uint32_t* clip;       // [n_tri] triangles that reach behind the near plane
  TilePair* pairs;      // [capacity]
  uint32_t* lists;      // [capacity] items by tile
  TileRecord* wide;     // [wide_capacity] what every tile looks at
  TileRecord* cut;      // [cut_capacity] what the lists hold of clipped triangles
};

// A triangle without room in the lists or the records.
__device__ __forceinline__ void leave_out(const TileArgs& a, uint32_t t) { a.r.big[atomicAdd(a.r.n_big, 1u)] = t; }
// A triangle's piece for every tile to look at; false: no room.
__device__ __forceinline__ bool add_wide(const TileArgs& a, const TileRecord& rec) {
  const uint32_t i = atomicAdd(&a.head[0], 1u);
  if (i < a.wide_capacity) a.wide[i] = rec;
  return i < a.wide_capacity;
}

__device__ __forceinline__ TileRecord tile_record(const Setup& st, uint32_t t, uint32_t piece) {
  const uint32_t x0 = st.px0 / kTile, x1 = (st.px0 + st.bw - 1) / kTile;
  const uint32_t y0 = st.py0 / kTile, y1 = (st.py0 + st.bh - 1) / kTile;
  return TileRecord{x0 | (x1 << 16), y0 | (y1 << 16), t, piece};
}

// Tiles of a piece if they are few enough for the lists, else 0.
__device__ __forceinline__ uint32_t list_tiles(const TileRecord& rec) {
  const uint32_t nx = (rec.x >> 16) - (rec.x & 0xffffu) + 1u, ny = (rec.y >> 16) - (rec.y & 0xffffu) + 1u;
  return nx > kTileSpan || ny > kTileSpan || nx * ny > kTileSpan ? 0u : nx * ny;
}

// Claimed pairs that stay unused because they pass the capacity.
__device__ __forceinline__ void drop_pairs(const TileArgs& a, uint32_t base, uint32_t n) {
  for (uint32_t i = base; i < a.capacity && i - base < n; ++i) a.pairs[i].tile = kNoTile;
}

// The pairs of the workgroup's triangles are spread over its threads again (a
// thread that walked its own triangle's tiles held up its wave: 130 us, this
// 47).  The neighbours in a mesh fall into the same tiles, so a wave adds up
// its pairs of a tile before its atomics (125 us with an atomic for each), whose
// results are the ranks that spare the fill a second round of them.
__global__ __launch_bounds__(1024) void k_tile_count(TileArgs a) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = __lane_id();
  uint32_t tiles = 0;
  TileRecord rec{};
  bool big = false;
  if (t < a.r.n_tri) {
    float p[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) p[i] = a.r.positions[9 * static_cast<size_t>(t) + i];
    ScreenTri sc;
    bool degenerate;
    const int front = project_front(p, a.r.vp, a.r.w, a.r.h, sc, degenerate);
    if (front == 1 || front == 2) {
      a.clip[atomicAdd(&a.head[1], 1u)] = t;
    } else if (front == 3 && !degenerate) {
      const Setup st = setup_piece(sc, a.r.w, a.r.h);
      if (st.ok) {
        rec = tile_record(st, t, 2u);
        tiles = list_tiles(rec);
        big = tiles == 0u;
      }
    }
  }
  // Where the thread's pairs end in the workgroup's.
  __shared__ uint32_t ends[1024], first_x[1024], first_y[1024], width[1024], wave_sum[16], group_base;
  uint32_t upto = tiles;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(upto, o);
    if (static_cast<int>(lane) >= o) upto += u;
  }
  const uint32_t w = threadIdx.x >> 6;
  if (lane == 63u) wave_sum[w] = upto;
  __syncthreads();
  uint32_t sum = 0u;
#pragma unroll
  for (uint32_t k = 0; k < 16u; ++k) {
    upto += k < w ? wave_sum[k] : 0u;
    sum += wave_sum[k];
  }
  if (threadIdx.x == 0u && sum != 0u) group_base = atomicAdd(&a.head[2], sum);
  ends[threadIdx.x] = upto;
  first_x[threadIdx.x] = rec.x & 0xffffu;
  first_y[threadIdx.x] = rec.y & 0xffffu;
  width[threadIdx.x] = (rec.x >> 16) - (rec.x & 0xffffu) + 1u;
  __syncthreads();
  bool out = big && !add_wide(a, rec);
  if (sum != 0u && (group_base > a.capacity || sum > a.capacity - group_base)) {
    if (threadIdx.x == 0u) drop_pairs(a, group_base, sum);
    out = out || tiles != 0u;
    sum = 0u;
  }
  if (out) leave_out(a, t);
  for (uint32_t i0 = 0; i0 < sum; i0 += 1024u) {
    // Pair i: the first thread whose pairs end behind it, then its tile.
    const uint32_t i = i0 + threadIdx.x;
    const bool on = i < sum;
    uint32_t owner = 0u;
#pragma unroll
    for (uint32_t step = 512u; step > 0u; step >>= 1) owner += on && ends[owner + step - 1u] <= i ? step : 0u;
    const uint32_t nx = width[owner], q = i - (owner != 0u ? ends[owner - 1u] : 0u);
    const uint32_t tile = (first_y[owner] + q / nx) * static_cast<uint32_t>(a.tiles_x) + first_x[owner] + q % nx;
    uint64_t left = __ballot(on);
    uint32_t leader = lane, rank = 0u, n = 1u;
    for (int k = 0; k < kTileGroups && left != 0ull; ++k) {
      const int first = __builtin_ctzll(left);
      const uint32_t its = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tile), first));
      const uint64_t same = __ballot(on && tile == its);
      if (on && tile == its) {
        leader = static_cast<uint32_t>(first);
        rank = static_cast<uint32_t>(__popcll(same & ((1ull << lane) - 1ull)));
        n = static_cast<uint32_t>(__popcll(same));
      }
      left &= ~same;
    }
    uint32_t before = 0u;
    if (on && leader == lane) before = atomicAdd(&a.count[tile], n);
    before = __shfl(before, static_cast<int>(leader));
    if (on) a.pairs[group_base + i] = TilePair{blockIdx.x * 1024u + owner, tile, before + rank};
  }
}

// The pieces of triangles cut by the near plane.
__global__ __launch_bounds__(256) void k_tile_clip(TileArgs a) {
  const uint32_t n = a.head[1];
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t t = a.clip[i];
    ScreenTri sc[2];
    const int m = project_clip(a.r.positions + 9 * static_cast<size_t>(t), a.r.vp, a.r.w, a.r.h, sc);
    bool out = false;  // whole, though one piece may be in the lists: the same fragments
    for (int k = 0; k < m; ++k) {
      const Setup st = setup_piece(sc[k], a.r.w, a.r.h);
      if (!st.ok) continue;
      const TileRecord rec = tile_record(st, t, static_cast<uint32_t>(k));
      const uint32_t tiles = list_tiles(rec);
      if (tiles == 0u) {
        out = !add_wide(a, rec) || out;
        continue;
      }
      uint32_t slot = atomicAdd(&a.head[2], tiles);
      const bool fits = slot <= a.capacity && tiles <= a.capacity - slot;
      const uint32_t r = fits ? atomicAdd(&a.head[3], 1u) : a.cut_capacity;
      if (r >= a.cut_capacity) {
        drop_pairs(a, slot, tiles);
        out = true;
        continue;
      }
      a.cut[r] = rec;
      for (uint32_t y = rec.y & 0xffffu; y <= rec.y >> 16; ++y)
        for (uint32_t x = rec.x & 0xffffu; x <= rec.x >> 16; ++x, ++slot) {
          const uint32_t tile = y * static_cast<uint32_t>(a.tiles_x) + x;
          a.pairs[slot] = TilePair{kRecordItem | r, tile, atomicAdd(&a.count[tile], 1u)};
        }
    }
    if (out) leave_out(a, t);
  }
}

// Where each tile's list begins, in any order of the tiles: a wave takes the room
// of its 64 at once (one workgroup that scanned all counts took 9 us at 1920x1080
// and 25 at 3840x2160).  The workgroups after those of the tiles empty the pixels
// if triangles are left to the two passes.
__global__ __launch_bounds__(256) void k_tile_start(TileArgs a) {
  const uint32_t n = static_cast<uint32_t>(a.tiles_x) * static_cast<uint32_t>(a.tiles_y), groups = (n + 255u) / 256u;
  if (blockIdx.x >= groups) {
    if (*a.r.n_big == 0u) return;
    const size_t pixels = static_cast<size_t>(a.r.w) * a.r.h, step = (gridDim.x - groups) * size_t(256);
    for (size_t i = (blockIdx.x - groups) * size_t(256) + threadIdx.x; i < pixels; i += step) {
      a.r.zbits[i] = 0ull;
      a.r.tri[i] = 0xffffffffu;
    }
    return;
  }
  const uint32_t i = blockIdx.x * 256u + threadIdx.x, lane = threadIdx.x & 63u;
  const uint32_t c = i < n ? a.count[i] : 0u;
  uint32_t upto = c;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(upto, o);
    if (static_cast<int>(lane) >= o) upto += u;
  }
  uint32_t base = 0u;
  if (lane == 63u) base = atomicAdd(&a.head[5], upto);
  base = __shfl(base, 63);
  if (i < n) a.start[i] = base + upto - c;
}

// The pairs into the tiles' lists, and the depth pass of the triangles left to
// the two passes.
__global__ __launch_bounds__(256) void k_tile_fill(TileArgs a) {
  const uint32_t n = min(a.head[2], a.capacity);
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const TilePair p = a.pairs[i];
    if (p.tile != kNoTile) a.lists[a.start[p.tile] + p.rank] = p.item;
  }
  raster_big(a.r, [&](uint32_t, size_t i, double z) {
    atomicMax(&a.r.zbits[i], static_cast<unsigned long long>(__double_as_longlong(z)));
  });
}

// A batch of triangles in LDS: what raster_piece reads, and FP32 planes
// a X + b Y + c over the tile's pixel centres (X, Y from the tile's corner) of
// the three edge functions and the depth, each raised above all rounding of
// the plane and of the FP64 test: below zero, or a depth plane below the depth
// held, is outside or behind for sure.  39 KB: four workgroups on a CU.
struct TilePrim {
  double x[3], y[3], z[3], inv;
};
struct TileBatch {
  TilePrim prim[256];
  float4 plane[3][256];
  uint2 box_tri[256];   // columns | rows << 16 of the tile inside the pixel box; index
  float zmax[4][256];   // above every depth in the wave's 8x8 pixels
  uint8_t touch[256];   // bit per wave: may cover a pixel of it
  uint16_t queue[512];  // wide records that touch the tile
  uint16_t found[4];
};
static_assert(sizeof(TileBatch) <= 40960, "four workgroups on a CU");

// g bounds the terms that c and the FP64 test were summed from.
__device__ __forceinline__ void tile_plane(float* out, double a, double b, double c, double g) {
  const double m = 16.0 * (fabs(a) + fabs(b)) + fabs(c);
  const double top = c + m * 0x1p-20 + g * 0x1p-40 + 1e-30;
  const bool usable = m < 1e30 && g < 1e30;  // false also for NaN
  out[0] = usable ? static_cast<float>(a) : 0.0f;
  out[1] = usable ? static_cast<float>(b) : 0.0f;
  out[2] = usable ? static_cast<float>(top) : 1e38f;
}

__device__ __forceinline__ float plane_at(float a, float b, float c, float x, float y) {
  return __builtin_fmaf(a, x, __builtin_fmaf(b, y, c));
}

// Thread tid's triangle of the batch; the waves that it may touch.
__device__ __forceinline__ uint32_t tile_prim(TileBatch& e, uint32_t tid, const ScreenTri& q, uint32_t t, int w, int h,
                                              int ox, int oy) {
  const Setup st = setup_piece(q, w, h);
  if (!st.ok) return 0u;
  const int x0 = max(st.px0 - ox, 0), x1 = min(st.px0 + st.bw - 1 - ox, kTile - 1);
  const int y0 = max(st.py0 - oy, 0), y1 = min(st.py0 + st.bh - 1 - oy, kTile - 1);
  if (x0 > x1 || y0 > y1) return 0u;
  const double a0 = -(q.y[2] - q.y[1]) * st.inv, b0 = (q.x[2] - q.x[1]) * st.inv;
  const double a1 = -(q.y[0] - q.y[2]) * st.inv, b1 = (q.x[0] - q.x[2]) * st.inv;
  const double rx1 = ox - q.x[1], ry1 = oy - q.y[1], rx2 = ox - q.x[2], ry2 = oy - q.y[2];
  const double c0 = b0 * ry1 + a0 * rx1, c1 = b1 * ry2 + a1 * rx2;
  const double g0 = fabs(b0) * (fabs(ry1) + 16.0) + fabs(a0) * (fabs(rx1) + 16.0);
  const double g1 = fabs(b1) * (fabs(ry2) + 16.0) + fabs(a1) * (fabs(rx2) + 16.0);
  const double u = q.z[0] - q.z[2], v = q.z[1] - q.z[2];
  const double zsum = fabs(q.z[0]) + fabs(q.z[1]) + fabs(q.z[2]);
  float p[12];
  tile_plane(p + 0, a0, b0, c0, g0);
  tile_plane(p + 3, a1, b1, c1, g1);
  tile_plane(p + 6, -(a0 + a1), -(b0 + b1), 1.0 - c0 - c1, 1.0 + g0 + g1);
  tile_plane(p + 9, a0 * u + a1 * v, b0 * u + b1 * v, c0 * u + c1 * v + q.z[2], (1.0 + g0 + g1) * zsum);
  const double top = fmax(fmax(q.z[0], q.z[1]), q.z[2]) + zsum * 0x1p-20 + 1e-30;
  const float zmax = top < 1e30 ? static_cast<float>(top) : 1e38f;
  uint32_t touch = 0u;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int kx = 8 * (k & 1), ky = 8 * (k >> 1);
    // Each plane at the pixel centre of the 8x8 where it is greatest.
    bool in = x0 < kx + 8 && x1 >= kx && y0 < ky + 8 && y1 >= ky;
    float at[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      at[c] = plane_at(p[3 * c], p[3 * c + 1], p[3 * c + 2], static_cast<float>(kx) + (p[3 * c] > 0.0f ? 7.5f : 0.5f),
                       static_cast<float>(ky) + (p[3 * c + 1] > 0.0f ? 7.5f : 0.5f));
    in = in && !(at[0] < 0.0f) && !(at[1] < 0.0f) && !(at[2] < 0.0f) && !(at[3] < 0.0f);
    touch |= in ? 1u << k : 0u;
    e.zmax[k][tid] = fminf(zmax, at[3]);
  }
  TilePrim& d = e.prim[tid];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    d.x[k] = q.x[k];
    d.y[k] = q.y[k];
    d.z[k] = q.z[k];
    e.plane[k][tid] = make_float4(p[4 * k], p[4 * k + 1], p[4 * k + 2], p[4 * k + 3]);
  }
  d.inv = st.inv;
  e.box_tri[tid] = make_uint2((((2u << (x1 - x0)) - 1u) << x0) | ((((2u << (y1 - y0)) - 1u) << y0) << 16), t);
  return touch;
}

__global__ __launch_bounds__(256, 4) void k_tile_raster(TileArgs a) {
  __shared__ TileBatch e;
  const int tile_x = static_cast<int>(blockIdx.x) % a.tiles_x, tile_y = static_cast<int>(blockIdx.x) / a.tiles_x;
  const int ox = tile_x * kTile, oy = tile_y * kTile;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lx = (lane & 7u) + 8u * (w & 1u), ly = (lane >> 3) + 8u * (w >> 1);
  const int px = ox + static_cast<int>(lx), py = oy + static_cast<int>(ly);
  const bool inside = px < a.r.w && py < a.r.h;
  const double cx = px + 0.5, cy = py + 0.5;
  const float fx = static_cast<float>(lx) + 0.5f, fy = static_cast<float>(ly) + 0.5f;
  const uint32_t bit = (1u << lx) | (0x10000u << ly);
  double z = 0.0;                      // a fragment must beat the cleared depth 0
  uint32_t id = 0xffffffffu;
  const size_t pixel = static_cast<size_t>(py) * a.r.w + px;
  if (*a.r.n_big != 0u && inside) {  // what the two passes drew
    z = __longlong_as_double(static_cast<long long>(a.r.zbits[pixel]));
    id = a.r.tri[pixel];
  }
  float zlow = inside ? static_cast<float>(z) * (1.0f - 0x1p-20f) : 1e38f;  // below z

  // First the wide records, gathered to whole batches, then the tile's list.
  const uint32_t n_wide = min(a.head[0], a.wide_capacity);
  const uint32_t begin = a.start[blockIdx.x], n_list = a.count[blockIdx.x];
  uint32_t looked = 0u, queued = 0u, taken = 0u;
  while (looked < n_wide || queued != 0u || taken < n_list) {
    while (looked < n_wide && queued < 256u) {
      const uint32_t i = looked + tid;
      bool hit = i < n_wide;
      if (hit) {
        const TileRecord rec = a.wide[i];
        const uint32_t tx = static_cast<uint32_t>(tile_x), ty = static_cast<uint32_t>(tile_y);
        hit = tx >= (rec.x & 0xffffu) && tx <= (rec.x >> 16) && ty >= (rec.y & 0xffffu) && ty <= (rec.y >> 16);
      }
      looked += 256u;
      if (!__syncthreads_or(hit)) continue;
      const uint64_t hits = __ballot(hit);
      if (lane == 0u) e.found[w] = static_cast<uint16_t>(__popcll(hits));
      __syncthreads();
      uint32_t at = queued + static_cast<uint32_t>(__popcll(hits & ((1ull << lane) - 1ull)));
#pragma unroll
      for (uint32_t k = 0; k < 4u; ++k) {
        at += k < w ? e.found[k] : 0u;
        queued += e.found[k];
      }
      if (hit) e.queue[at] = static_cast<uint16_t>(i);
      __syncthreads();
    }
    const uint32_t n_queue = min(queued, 256u), n_items = min(256u - n_queue, n_list - taken);
    const bool from_queue = tid < n_queue, valid = tid < n_queue + n_items;
    uint32_t item = 0u, piece = 2u;
    uint16_t left = 0u;
    if (valid) {
      if (!from_queue) item = a.lists[begin + taken + (tid - n_queue)];
      if (from_queue || (item & kRecordItem)) {
        const TileRecord rec = from_queue ? a.wide[e.queue[tid]] : a.cut[item & ~kRecordItem];
        item = rec.tri;
        piece = rec.piece;
      }
    }
    taken += n_items;
    if (queued > 256u) {  // what is left of the queue moves up
      left = e.queue[256u + tid];
      __syncthreads();
      e.queue[tid] = left;
    }
    queued -= n_queue;
    uint32_t touch = 0u;
    if (valid) {
      ScreenTri q;
      const float* pos = a.r.positions + 9 * static_cast<size_t>(item);
      if (piece == 2u) {
        float p[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) p[k] = pos[k];
        bool degenerate;
        project_front(p, a.r.vp, a.r.w, a.r.h, q, degenerate);
      } else {
        ScreenTri sc[2];
        project_clip(pos, a.r.vp, a.r.w, a.r.h, sc);
        q = piece ? sc[1] : sc[0];
      }
      touch = tile_prim(e, tid, q, item, a.r.w, a.r.h, ox, oy);
    }
    e.touch[tid] = static_cast<uint8_t>(touch);
    __syncthreads();
    for (uint32_t k = 0; k < 256u; k += 64u) {
      // The triangles that touch the wave's pixels and may lie before the farthest.
      float far = zlow;
      for (int o = 32; o > 0; o >>= 1) far = fminf(far, __shfl_xor(far, o));
      uint64_t todo = __ballot((e.touch[k + lane] >> w & 1u) != 0u && !(e.zmax[w][k + lane] < far));
      while (todo != 0ull) {
        const uint32_t j = k + static_cast<uint32_t>(__builtin_ctzll(todo));
        todo &= todo - 1ull;
        const uint2 bt = e.box_tri[j];
        const float4 p0 = e.plane[0][j], p1 = e.plane[1][j], p2 = e.plane[2][j];
        const bool maybe = ((bt.x & bit) == bit) & !(plane_at(p0.x, p0.y, p0.z, fx, fy) < 0.0f) &
                           !(plane_at(p0.w, p1.x, p1.y, fx, fy) < 0.0f) & !(plane_at(p1.z, p1.w, p2.x, fx, fy) < 0.0f) &
                           !(plane_at(p2.y, p2.z, p2.w, fx, fy) < zlow);
        if (__ballot(maybe) == 0ull) continue;
        const TilePrim& q = e.prim[j];
        const double e0 = ((q.x[2] - q.x[1]) * (cy - q.y[1]) - (q.y[2] - q.y[1]) * (cx - q.x[1])) * q.inv;
        const double e1 = ((q.x[0] - q.x[2]) * (cy - q.y[2]) - (q.y[0] - q.y[2]) * (cx - q.x[2])) * q.inv;
        const double e2 = 1.0 - e0 - e1;
        const double f = e0 * q.z[0] + e1 * q.z[1] + e2 * q.z[2];
        const bool hit = maybe && !(e0 < 0 || e1 < 0 || e2 < 0) && f > 0.0 && !(f > 1.0);
        if (hit && (f > z || (f == z && bt.y < id))) {
          z = f;
          id = bt.y;
          zlow = static_cast<float>(f) * (1.0f - 0x1p-20f);
        }
      }
    }
    __syncthreads();
  }
  if (!inside) return;
  a.r.zbits[pixel] = static_cast<unsigned long long>(__double_as_longlong(z));
  a.r.tri[pixel] = id;
}

// ---- formats (bit-exact restatements of the host producer's) ------------

__device__ uint16_t f32_to_f16(float f) {
  const uint32_t x = __float_as_uint(f);
  const uint32_t sign = (x >> 16) & 0x8000u;
  uint32_t mant = x & 0x7fffffu;
  const int exp = static_cast<int>((x >> 23) & 0xffu);
  if (exp == 0xff) return static_cast<uint16_t>(sign | 0x7c00u | (mant ? 0x200u : 0u));
  const int e = exp - 127 + 15;
  if (e >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
  if (e <= 0) {
    if (e < -10) return static_cast<uint16_t>(sign);
    mant |= 0x800000u;
    const int shift = 14 - e;
    uint32_t h = mant >> shift;
    const uint32_t rem = mant & ((1u << shift) - 1u);
    const uint32_t half = 1u << (shift - 1);
    if (rem > half || (rem == half && (h & 1u))) ++h;
    return static_cast<uint16_t>(sign | h);
  }
  uint32_t h = (static_cast<uint32_t>(e) << 10) | (mant >> 13);
  const uint32_t rem = mant & 0x1fffu;
  if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) ++h;
  return static_cast<uint16_t>(sign | h);
}

__device__ __forceinline__ int16_t clamp_i16(float v) {
  // GLSL int() truncation, then the RG16I store (saturating).
  const int i = to_int(v);
  return static_cast<int16_t>(min(32767, max(-32768, i)));
}

// PackNormal16I, shader/utils.glsl:65-89.
__device__ __forceinline__ void pack_normal16i(const float* n, int16_t* out) {
  const float px = (n[0] == 0.0f) ? ((n[1] > 0.0f ? 1.0f : (n[1] < 0.0f ? -1.0f : 0.0f)) * kPiF / 2.0f)
                                  : atan2f(n[1], n[0]);
  out[0] = clamp_i16(px * (32768.0f / kPiF));
  out[1] = clamp_i16(n[2] * 32768.0f);
}

__device__ __forceinline__ uint8_t srgb_encode(float c) {
  c = fminf(1.0f, fmaxf(0.0f, c));
  // Settled in FP32 unless the value lies near a step: the hardware's log2 and
  // exp2 keep 255 s within 2e-4 (equal for every float in [0, 1]).
  const float q = c <= 0.0031308f ? 12.92f * c
                                  : 1.055f * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(c) * (1.0f / 2.4f)) - 0.055f;
  const float v = q * 255.0f + 0.5f, low = floorf(v);
  if (v - low > 0.002f && v - low < 0.998f) return static_cast<uint8_t>(low);
  const double s = c <= 0.0031308 ? 12.92 * c : 1.055 * pow(static_cast<double>(c), 1.0 / 2.4) - 0.055;
  return static_cast<uint8_t>(floor(s * 255.0 + 0.5));
}

// ---- resolves -----------------------------------------------------------

struct GbufArgs {
  int w, h;
  const unsigned long long* zbits;
  const uint32_t* tri;
  const float* albedo;
  const float* normals;
  float* depth;
  int16_t* normal;
  uint8_t* albedo_srgb;
};

// shader/fillgbuffer.frag: depth, packed normal, sRGB albedo.  A thread shades
// four pixels, so that every texture is read and written in words (a pixel and
// three byte stores for each thread, with pow in FP64: 38 us at 1920x1080, now 22).
__device__ __forceinline__ void shade_gbuffer(const GbufArgs& a, uint32_t t, int16_t* n, uint8_t* al) {
  n[0] = n[1] = 0;
  al[0] = al[1] = al[2] = 0;
  if (t == 0xffffffffu) return;
  pack_normal16i(a.normals + 3 * static_cast<size_t>(t), n);
#pragma unroll
  for (int k = 0; k < 3; ++k) al[k] = srgb_encode(a.albedo[3 * static_cast<size_t>(t) + k]);
}

__global__ __launch_bounds__(256) void k_gbuffer_resolve(GbufArgs a) {
  const size_t i = 4 * (static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x);
  const size_t n = static_cast<size_t>(a.w) * a.h;
  if (i >= n) return;
  if (i + 4 > n) {
    for (size_t p = i; p < n; ++p) {
      a.depth[p] = static_cast<float>(__longlong_as_double(static_cast<long long>(a.zbits[p])));
      shade_gbuffer(a, a.tri[p], a.normal + 2 * p, a.albedo_srgb + 3 * p);
    }
    return;
  }
  const uint4 t4 = *reinterpret_cast<const uint4*>(a.tri + i);
  const double2 z0 = *reinterpret_cast<const double2*>(a.zbits + i), z1 = *reinterpret_cast<const double2*>(a.zbits + i + 2);
  *reinterpret_cast<float4*>(a.depth + i) = make_float4(static_cast<float>(z0.x), static_cast<float>(z0.y),
                                                        static_cast<float>(z1.x), static_cast<float>(z1.y));
  const uint32_t t[4] = {t4.x, t4.y, t4.z, t4.w};
  uint32_t nw[4], aw[3] = {0u, 0u, 0u};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int16_t nn[2];
    uint8_t al[3];
    shade_gbuffer(a, t[k], nn, al);
    nw[k] = static_cast<uint16_t>(nn[0]) | (static_cast<uint32_t>(static_cast<uint16_t>(nn[1])) << 16);
#pragma unroll
    for (int c = 0; c < 3; ++c) aw[(3 * k + c) / 4] |= static_cast<uint32_t>(al[c]) << (8 * ((3 * k + c) % 4));
  }
  *reinterpret_cast<uint4*>(a.normal + 2 * i) = make_uint4(nw[0], nw[1], nw[2], nw[3]);
  uint32_t* out = reinterpret_cast<uint32_t*>(a.albedo_srgb + 3 * i);
  out[0] = aw[0];
  out[1] = aw[1];
  out[2] = aw[2];
}

struct RsmArgs {
  int res;
  const unsigned long long* zbits;
  const uint32_t* tri;
  const float* albedo;
  const float* normals;
  double ivp[16];
  float light_pos[3], light_dir[3], intensity[3];
  float cos_half;
  uint16_t* flux;
  int16_t* normal;
  uint16_t* dls;
  float* shadow;  // the light's depth buffer (the direct-lighting shadow map)
};

// shader/fillrsm.frag:32-61 at one texel: flux = albedo * I * spot falloff *
// pixel solid angle / pi, the packed normal, and (d, d^2) of the distance
// to the light; the world position is reconstructed from the depth.
__global__ __launch_bounds__(256) void k_rsm_resolve(RsmArgs a) {
  const int res = a.res;
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<size_t>(res) * res) return;
  const int x = static_cast<int>(i % res), y = static_cast<int>(i / res);
  const uint32_t t = a.tri[i];
  a.shadow[i] = static_cast<float>(__longlong_as_double(static_cast<long long>(a.zbits[i])));
  if (t == 0xffffffffu) {
    a.flux[3 * i] = a.flux[3 * i + 1] = a.flux[3 * i + 2] = 0;
    a.normal[2 * i] = a.normal[2 * i + 1] = 0;
    a.dls[2 * i] = a.dls[2 * i + 1] = 0;
    return;
  }
  const float d = static_cast<float>(__longlong_as_double(static_cast<long long>(a.zbits[i])));
  const double ndc[4] = {(x + 0.5) / res * 2.0 - 1.0, (y + 0.5) / res * 2.0 - 1.0, static_cast<double>(d), 1.0};
  double wp[4];
  for (int r = 0; r < 4; ++r)
    wp[r] = a.ivp[4 * r] * ndc[0] + a.ivp[4 * r + 1] * ndc[1] + a.ivp[4 * r + 2] * ndc[2] + a.ivp[4 * r + 3];
  const float pos[3] = {static_cast<float>(wp[0] / wp[3]), static_cast<float>(wp[1] / wp[3]),
                        static_cast<float>(wp[2] / wp[3])};
  float tl[3] = {a.light_pos[0] - pos[0], a.light_pos[1] - pos[1], a.light_pos[2] - pos[2]};
  const float dist = sqrtf(tl[0] * tl[0] + tl[1] * tl[1] + tl[2] * tl[2]);
  for (float& v : tl) v /= dist;
  float cos_to_light = -(tl[0] * a.light_dir[0] + tl[1] * a.light_dir[1] + tl[2] * a.light_dir[2]);
  cos_to_light = fminf(1.0f, fmaxf(0.0f, cos_to_light));
  const float total_sr = kPi2F * (1.0f - a.cos_half);
  const float pixel_sr = total_sr * cos_to_light / static_cast<float>(res) / static_cast<float>(res);
  const float falloff = fminf(1.0f, fmaxf(0.0f, cos_to_light - a.cos_half)) / (1.0f - a.cos_half);
  for (int k = 0; k < 3; ++k)
    a.flux[3 * i + k] = f32_to_f16(a.albedo[3 * static_cast<size_t>(t) + k] * a.intensity[k] * (falloff * pixel_sr / kPiF));
  a.dls[2 * i] = f32_to_f16(dist);
  a.dls[2 * i + 1] = f32_to_f16(dist * dist);
  pack_normal16i(a.normals + 3 * static_cast<size_t>(t), a.normal + 2 * i);
}

// One texel of a level as it is stored.
struct RsmTexel {
  uint16_t flux[3];
  int16_t normal[2];
  uint16_t dls[2];
};

// shader/downsamplersm.frag:15-33: flux summed over 2x2, normal the
// normalized mean repacked, (d, d^2) averaged.
__device__ __forceinline__ RsmTexel downsample(const RsmTexel* s) {
  RsmTexel o;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float a = half_to_float(s[0].flux[k]) + half_to_float(s[1].flux[k]);
    const float b = half_to_float(s[2].flux[k]) + half_to_float(s[3].flux[k]);
    o.flux[k] = f32_to_f16(a + b);
  }
  float n[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f3 u = unpack_normal16i(s[j].normal[0], s[j].normal[1]);
    n[0] += u.x;
    n[1] += u.y;
    n[2] += u.z;
  }
  const float l = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
  if (l > 0.0f)
    for (float& v : n) v /= l;
  pack_normal16i(n, o.normal);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float a = half_to_float(s[0].dls[k]) + half_to_float(s[1].dls[k]);
    const float b = half_to_float(s[2].dls[k]) + half_to_float(s[3].dls[k]);
    o.dls[k] = f32_to_f16((a + b) * 0.25f);
  }
  return o;
}

// Up to kRsmLevels levels above the level of res^2 texels at the start of the
// textures: a workgroup takes a square of 2^levels texels a side and keeps each
// level in LDS for the next (a launch for each level of a 256^2 RSM took 50 us,
// two launches 27; the time is the chain of sine, cosine and arc tangent).
constexpr int kRsmLevels = 5;

__global__ __launch_bounds__(256) void k_rsm_downsample(int res, int levels, uint16_t* flux, int16_t* normal,
                                                        uint16_t* dls) {
  __shared__ RsmTexel tile[2][256];
  const int across = res >> levels;
  const int bx = static_cast<int>(blockIdx.x) % across, by = static_cast<int>(blockIdx.x) / across;
  const int t = static_cast<int>(threadIdx.x);
  size_t off = 0;  // of the level below, in texels
  for (int l = 1; l <= levels; ++l) {
    const int lb = levels - l, side = 1 << lb, r = res >> (l - 1), r2 = r / 2;
    const size_t next = off + static_cast<size_t>(r) * r;
    if (t < side * side) {
      const int x = t & (side - 1), y = t >> lb;
      RsmTexel s[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int sx = 2 * x + (j & 1), sy = 2 * y + (j >> 1);
        if (l == 1) {
          const size_t p = off + static_cast<size_t>(by * 2 * side + sy) * r + (bx * 2 * side + sx);
          for (int k = 0; k < 3; ++k) s[j].flux[k] = flux[3 * p + k];
          for (int k = 0; k < 2; ++k) s[j].normal[k] = normal[2 * p + k];
          for (int k = 0; k < 2; ++k) s[j].dls[k] = dls[2 * p + k];
        } else {
          s[j] = tile[l & 1][sy * 2 * side + sx];
        }
      }
      const RsmTexel o = downsample(s);
      tile[(l + 1) & 1][t] = o;
      const size_t p = next + static_cast<size_t>(by * side + y) * r2 + (bx * side + x);
      for (int k = 0; k < 3; ++k) flux[3 * p + k] = o.flux[k];
      for (int k = 0; k < 2; ++k) normal[2 * p + k] = o.normal[k];
      for (int k = 0; k < 2; ++k) dls[2 * p + k] = o.dls[k];
    }
    __syncthreads();
    off = next;
  }
}

// Depth and winning triangle of every pixel into zbits / tri; work: the
// raster's lists, of raster_work_words or else for two passes.
void raster(const float* positions, uint32_t n_tri, const float* vp, int w, int h, unsigned long long* zbits,
            uint32_t* tri, uint32_t* work, size_t work_words, hipStream_t s) {
  RasterArgs a;
  a.positions = positions;
  a.n_tri = n_tri;
  for (int i = 0; i < 16; ++i) a.vp[i] = vp[i];
  a.w = w;
  a.h = h;
  a.zbits = zbits;
  a.tri = tri;
  a.n_big = work;  // work[0] counts, the list follows
  a.big = work + 1;
  const dim3 grid((n_tri + 255) / 256);
  if (tiled(w, h, n_tri) && work_words >= raster_work_words(w, h, n_tri)) {
    TileArgs t;
    t.r = a;
    t.tiles_x = (w + kTile - 1) / kTile;
    t.tiles_y = (h + kTile - 1) / kTile;
    const size_t tiles = static_cast<size_t>(t.tiles_x) * t.tiles_y, n = n_tri;
    const TileRoom room = tile_room(w, h, n_tri);
    t.capacity = room.pairs;
    t.wide_capacity = room.wide;
    t.cut_capacity = room.cut;
    t.wide = reinterpret_cast<TileRecord*>(work);
    t.cut = t.wide + room.wide;
    t.head = reinterpret_cast<uint32_t*>(t.cut + room.cut);
    t.count = t.head + kHeadWords;
    t.start = t.count + tiles;
    t.clip = t.start + tiles;
    t.lists = t.clip + n;
    t.pairs = reinterpret_cast<TilePair*>(t.lists + t.capacity);
    t.r.n_big = t.head + 4;
    t.r.big = reinterpret_cast<uint32_t*>(t.pairs + t.capacity);
    launch_fill_u32(t.head, kHeadWords + tiles, 0u, s);
    if (n_tri != 0) {
      hipLaunchKernelGGL(k_tile_count, dim3((n_tri + 1023) / 1024), dim3(1024), 0, s, t);
      hipLaunchKernelGGL(k_tile_clip, dim3(256), dim3(256), 0, s, t);
    }
    hipLaunchKernelGGL(k_tile_start, dim3(static_cast<unsigned>((tiles + 255) / 256) + (room.all ? 0 : 1024)), dim3(256), 0, s, t);
    if (n_tri != 0) hipLaunchKernelGGL(k_tile_fill, dim3(1024), dim3(256), 0, s, t);
    if (!room.all) hipLaunchKernelGGL(k_raster_id_big, dim3(1024), dim3(256), 0, s, t.r);
    hipLaunchKernelGGL(k_tile_raster, dim3(static_cast<unsigned>(tiles)), dim3(256), 0, s, t);
    return;
  }
  const size_t n = static_cast<size_t>(w) * h;
  hipLaunchKernelGGL(k_raster_clear, dim3(static_cast<unsigned>(std::min<size_t>((n + 255) / 256, 8192))), dim3(256), 0,
                     s, a);
  if (n_tri == 0) return;
  hipLaunchKernelGGL(k_raster_depth, grid, dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_raster_depth_big, dim3(1024), dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_raster_id, grid, dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_raster_id_big, dim3(1024), dim3(256), 0, s, a);
}

}  // namespace

void launch_render_gbuffer(const float* positions, const float* albedo, const float* normals, uint32_t n_tri,
                           const float* view_proj, int w, int h, unsigned long long* zbits, uint32_t* tri,
                           uint32_t* work, size_t work_words, float* depth, int16_t* normal, uint8_t* albedo_srgb,
                           hipStream_t s) {
  raster(positions, n_tri, view_proj, w, h, zbits, tri, work, work_words, s);
  GbufArgs a;
  a.w = w;
  a.h = h;
  a.zbits = zbits;
  a.tri = tri;
  a.albedo = albedo;
  a.normals = normals;
  a.depth = depth;
  a.normal = normal;
  a.albedo_srgb = albedo_srgb;
  const size_t n = static_cast<size_t>(w) * h;
  hipLaunchKernelGGL(k_gbuffer_resolve, dim3((n + 1023) / 1024), dim3(256), 0, s, a);
}

void launch_render_rsm(const float* positions, const float* albedo, const float* normals, uint32_t n_tri,
                       const drv_spot_light& light, unsigned long long* zbits, uint32_t* tri, uint32_t* work,
                       size_t work_words, uint16_t* flux, int16_t* normal, uint16_t* dls, float* shadow,
                       hipStream_t s) {
  const int res = light.rsm_render_resolution;
  raster(positions, n_tri, light.light_view_projection, res, res, zbits, tri, work, work_words, s);
  RsmArgs a;
  a.res = res;
  a.zbits = zbits;
  a.tri = tri;
  a.albedo = albedo;
  a.normals = normals;
  for (int i = 0; i < 16; ++i) a.ivp[i] = light.inverse_light_view_projection[i];
  for (int i = 0; i < 3; ++i) {
    a.light_pos[i] = light.light_position[i];
    a.light_dir[i] = light.light_direction[i];
    a.intensity[i] = light.light_intensity[i];
  }
  a.cos_half = light.light_cos_half_angle;
  a.flux = flux;
  a.normal = normal;
  a.dls = dls;
  a.shadow = shadow;
  const size_t n = static_cast<size_t>(res) * res;
  hipLaunchKernelGGL(k_rsm_resolve, dim3((n + 255) / 256), dim3(256), 0, s, a);
  // Mip chain: level l + 1 from level l, packed one after another.
  size_t off = 0;
  int left = __builtin_ctz(static_cast<unsigned>(res));
  for (int r = res; left > 0;) {
    const int levels = std::min(left, kRsmLevels), across = r >> levels;
    hipLaunchKernelGGL(k_rsm_downsample, dim3(static_cast<unsigned>(across) * across), dim3(256), 0, s, r, levels,
                       flux + 3 * off, normal + 2 * off, dls + 2 * off);
    for (int l = 0; l < levels; ++l, r /= 2) off += static_cast<size_t>(r) * r;
    left -= levels;
  }
}

}  // namespace drvk
