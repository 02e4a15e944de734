// Stage B: scene voxelization, temporal blend and the voxel mip chain.
//
// Restates Voxelization::VoxelizeScene (rendering/voxelization.cpp:90-176):
// the conservative raster pass shader/voxelize.{vert,geom,frag}, the blend
// shader/voxelblend.comp:8-18 and the mip loop shader/voxelmipmap.comp:8-12.
//
// MI355X design: the geometry-shader raster becomes one thread per
// triangle (several for small scenes) that evaluates the geometry shader's
// pushed-out edge planes and depth plane directly and walks the covered pixels
// of its dominant-axis projection; the blend is a flat byte stream; each mip
// level is an exact integer 2x2x2 mean.  After the mips a "corner-expanded" copy
// of every level holds the 8 texels of each trilinear footprint as one 16-byte
// record, so the cone tracer issues one load per level instead of eight byte
// gathers.
#include <algorithm>

#include "drv_internal.hpp"
#include "k_common.hpp"

namespace drvk {
namespace {

// A small scene's triangles share the chip's lanes, up to 32 for each triangle
// as long as there are at most this many (the chip's wavefront slots); the
// set-up is repeated in each.  2176 triangles of 35 box pixels in
// 64^3: 36 us with a lane each, 5.3 us with 32 (64: 6.6); 152k triangles in 128^3:
// 19.8 with one, 13.0 with two (four: 14.2); 1.0M keep one.
constexpr uint64_t kVoxelizeLanes = 1u << 19;
constexpr int kVoxelizeShareLog2 = 5;

struct VoxelizeArgs {
  float vmin[3], vmax[3];
  float world[16];
  const float* positions;
  const uint32_t* indices;
  uint32_t n_tri;
  int res;
  int lanes_log2;  // lanes that share a triangle's pixels
  uint8_t* target;
};

__device__ __forceinline__ void store_voxel(uint8_t* target, int res, int side, int sx, int sy, int sz) {
  // UnswizzlePos, voxelize.frag:16-19
  int x, y, z;
  if (side == 0) {
    x = sz; y = sy; z = sx;
  } else if (side == 1) {
    x = sx; y = sz; z = sy;
  } else {
    x = sx; y = sy; z = sz;
  }
  // imageStore outside the image has no effect.
  if (x < 0 || y < 0 || z < 0 || x >= res || y >= res || z >= res) return;
  target[static_cast<uint32_t>((z * res + y) * res + x)] = 255;  // res <= 512
}

__global__ __launch_bounds__(256) void k_voxelize(VoxelizeArgs a) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t t = g >> a.lanes_log2, lanes = 1u << a.lanes_log2, sub = g & (lanes - 1u);
  if (t >= a.n_tri) return;
  const int res = a.res;
  const float fres = static_cast<float>(res);
  const float h = 1.0f / fres;
  // voxelize.vert:15-23
  float P[3][3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const uint32_t vi = a.indices ? a.indices[3 * t + v] : 3 * t + v;
    const float* p = a.positions + 3 * static_cast<size_t>(vi);
    float w4[4];
    mat_vec(a.world, p[0], p[1], p[2], 1.0f, w4);
#pragma unroll
    for (int i = 0; i < 3; ++i) P[v][i] = (w4[i] - a.vmin[i]) / (a.vmax[i] - a.vmin[i]) * 2.0f - 1.0f;
  }
  // voxelize.geom:43-48: dominant axis of the (normalized) face normal
  const float v0x = P[1][0] - P[0][0], v0y = P[1][1] - P[0][1], v0z = P[1][2] - P[0][2];
  const float v1x = P[2][0] - P[0][0], v1y = P[2][1] - P[0][1], v1z = P[2][2] - P[0][2];
  const float c0 = v0y * v1z - v0z * v1y, c1 = v0z * v1x - v0x * v1z, c2 = v0x * v1y - v0y * v1x;
  const float cl = sqrtf(c0 * c0 + c1 * c1 + c2 * c2);
  const float an0 = fabsf(c0 / cl), an1 = fabsf(c1 / cl), an2 = fabsf(c2 / cl);
  int side = an0 > an1 ? 0 : 1;
  side = (side == 0 ? an0 : an1) > an2 ? side : 2;
  // voxelize.geom:53-75: swizzle into the raster plane
  float r[3][3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    if (side == 0) {
      r[v][0] = P[v][2]; r[v][1] = P[v][1]; r[v][2] = P[v][0];
    } else if (side == 1) {
      r[v][0] = P[v][0]; r[v][1] = P[v][2]; r[v][2] = P[v][1];
    } else {
      r[v][0] = P[v][0]; r[v][1] = P[v][1]; r[v][2] = P[v][2];
    }
  }
  // voxelize.geom:81-83: raster AABB grown by half a voxel, in pixels
  float bb0 = fminf(fminf(r[0][0], r[1][0]), r[2][0]) - h;
  float bb1 = fminf(fminf(r[0][1], r[1][1]), r[2][1]) - h;
  float bb2 = fmaxf(fmaxf(r[0][0], r[1][0]), r[2][0]) + h;
  float bb3 = fmaxf(fmaxf(r[0][1], r[1][1]), r[2][1]) + h;
  bb0 = (bb0 * 0.5f + 0.5f) * fres;
  bb1 = (bb1 * 0.5f + 0.5f) * fres;
  bb2 = (bb2 * 0.5f + 0.5f) * fres;
  bb3 = (bb3 * 0.5f + 0.5f) * fres;
  // voxelize.geom:86-102: edge lines cross((d,0),(p,1)) = (d.y, -d.x, d.x p.y - d.y p.x),
  // oriented by the winding and pushed out by h * (|a| + |b|).
  const float ax = r[0][0] - r[2][0], ay = r[0][1] - r[2][1];
  const float bx = r[1][0] - r[0][0], by = r[1][1] - r[0][1];
  const float ex = r[2][0] - r[1][0], ey = r[2][1] - r[1][1];
  float pl[3][3] = {{ay, -ax, ax * r[2][1] - ay * r[2][0]},
                    {by, -bx, bx * r[0][1] - by * r[0][0]},
                    {ey, -ex, ex * r[1][1] - ey * r[1][0]}};
  const float wind_raw = ax * by - bx * ay;
  const float wind = wind_raw > 0.0f ? 1.0f : (wind_raw < 0.0f ? -1.0f : 0.0f);
  if (wind == 0.0f) return;  // zero-area primitive
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    pl[i][0] = pl[i][0] * wind;
    pl[i][1] = pl[i][1] * wind;
    pl[i][2] = pl[i][2] * wind;
    pl[i][2] = pl[i][2] - (h * fabsf(pl[i][0]) + h * fabsf(pl[i][1]));
  }
  // voxelize.geom:118-128: expanded vertices = pairwise line intersections,
  // each keeping its original depth.
  float V[3][3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const float* p = pl[v == 0 ? 0 : (v == 1 ? 1 : 2)];
    const float* q = pl[v == 0 ? 1 : (v == 1 ? 2 : 0)];
    const float cx = p[1] * q[2] - p[2] * q[1];
    const float cy = p[2] * q[0] - p[0] * q[2];
    const float cw = p[0] * q[1] - p[1] * q[0];
    V[v][0] = cx / cw;
    V[v][1] = cy / cw;
    V[v][2] = r[v][2];
  }
  const float ex1 = V[1][0] - V[0][0], ey1 = V[1][1] - V[0][1];
  const float ex2 = V[2][0] - V[0][0], ey2 = V[2][1] - V[0][1];
  const float area = ex1 * ey2 - ex2 * ey1;
  if (!(area != 0.0f) || !isfinite(area)) return;
  const float dz1 = V[1][2] - V[0][2], dz2 = V[2][2] - V[0][2];
  // dFdxCoarse / dFdyCoarse of gl_FragCoord.z * res == NDC depth gradient
  const float gx = (dz1 * ey2 - dz2 * ey1) / area;
  const float gy = (dz2 * ex1 - dz1 * ex2) / area;
  const float max_change = sqrtf(gx * gx + gy * gy) * 1.414f;
  // voxelize.frag:26-30 keeps the pixel centres c = p + 0.5 with
  // bb_lo <= c <= bb_hi, i.e. ceil(bb_lo - 0.5) <= p <= floor(bb_hi - 0.5).
  // bb - 0.5 is exact for bb >= 0.25 (Sterbenz up to 1, on bb's grid above);
  // a bound below 0.5 only ever yields p <= 0 (lower) or p < 0 (upper), as
  // the exact value does, so the ranges hold exactly the passing centres.
  const int px0 = max(0, to_int(ceilf(bb0 - 0.5f)));
  const int py0 = max(0, to_int(ceilf(bb1 - 0.5f)));
  const int px1 = min(res - 1, to_int(floorf(bb2 - 0.5f)));
  const int py1 = min(res - 1, to_int(floorf(bb3 - 0.5f)));
  if (px0 > px1 || py0 > py1) return;
  // The box's pixels in rows; this lane takes number sub, sub + lanes, ...
  const uint32_t bw = static_cast<uint32_t>(px1 - px0 + 1);
  int px = px0, py = py0;
  int cols = bw == 1u ? 0 : 1, rows = bw == 1u ? 1 : 0;
  if (lanes != 1u) {
    px += static_cast<int>(sub % bw);
    py += static_cast<int>(sub / bw);
    cols = static_cast<int>(lanes % bw);
    rows = static_cast<int>(lanes / bw);
  }
  // res is a power of two, so x / res == x * h exactly.
  while (py <= py1) {
    const float nx = (static_cast<float>(px) + 0.5f) * h * 2.0f - 1.0f;
    const float ny = (static_cast<float>(py) + 0.5f) * h * 2.0f - 1.0f;
    const bool in = (pl[0][0] * nx + pl[0][1] * ny + pl[0][2] <= 0.0f) &&
                    (pl[1][0] * nx + pl[1][1] * ny + pl[1][2] <= 0.0f) &&
                    (pl[2][0] * nx + pl[2][1] * ny + pl[2][2] <= 0.0f);
    if (in) {
      const float zn = V[0][2] + gx * (nx - V[0][0]) + gy * (ny - V[0][1]);
      const float zw = zn * 0.5f + 0.5f;
      // voxelize.frag:33-56
      const float vz = zw * fres;
      const int iz = to_int(vz);
      store_voxel(a.target, res, side, px, py, iz);
      if (iz != to_int(vz - max_change)) store_voxel(a.target, res, side, px, py, iz - 1);
      if (iz != to_int(vz + max_change)) store_voxel(a.target, res, side, px, py, iz + 1);
    }
    px += cols;
    py += rows;
    if (px > px1) {
      px -= static_cast<int>(bw);
      ++py;
    }
  }
}

// voxelblend.comp:8-18 (old + sign(target - old) * AdaptionFactor, stored as
// unorm8) and voxelmipmap.comp:8-12 (the linear sample at the centre of each
// 2x2x2 child block is the 8-texel mean, computed exactly and rounded half
// up), fused: one workgroup per slab of level 0, one to four 16^3 bricks along
// x, blends its texels and builds the bricks' levels 1..4 in LDS; the first
// workgroup of k_voxel_corners then builds the levels above from the bricks'
// top texels.
constexpr int kBrick = 16;

struct MipArgs {
  const uint8_t* target;
  uint8_t* mips;
  uint32_t mip_offset[16];
  int res, levels;
  int brick, brick_levels;  // B = min(16, res), log2(B)
  int slab_log2;            // log2 of the slab's texels along x
  float f;
};

// x / 255 correctly rounded, for whole x in [0, 255].
__device__ __forceinline__ float unorm8(uint32_t x) {
  const float t = static_cast<float>(x), r = 1.0f / 255.0f;
  const float q = t * r;
  return __builtin_fmaf(__builtin_fmaf(-255.0f, q, t), r, q);
}

// voxelblend.comp:8-18: old + sign(target - old) * AdaptionFactor, unorm8.
__device__ __forceinline__ uint8_t blend_voxel(uint32_t target, uint32_t old, float f) {
  const float tv = unorm8(target), o = unorm8(old);
  const float d = tv - o;
  const float sg = d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f);
  float v = o + sg * f;
  v = fminf(1.0f, fmaxf(0.0f, v));
  return static_cast<uint8_t>(floorf(v * 255.0f + 0.5f));
}

__device__ __forceinline__ uint8_t mean8(const uint8_t* s, int w, int x, int y, int z) {
  const uint8_t* s0 = s + (static_cast<size_t>(2 * z) * w + 2 * y) * w + 2 * x;
  const uint8_t* s1 = s0 + static_cast<size_t>(w) * w;
  const int sum = s0[0] + s0[1] + s0[w] + s0[w + 1] + s1[0] + s1[1] + s1[w] + s1[w + 1];
  return static_cast<uint8_t>((sum + 4) >> 3);
}

// Dynamic LDS: the slab's levels.  Bound by the texel rows' addresses: a brick
// alone has rows of 16 bytes, a line access for every lane, so a slab has up to
// four, as long as there is a workgroup for every CU.  Empty rows (most of a
// volume) skip the blend, unchanged ones the store.  256^3: 67 us with a
// workgroup per brick and divisions by 255 in every texel, 38 us; 128^3: 12 and
// 6.5 us.
__global__ __launch_bounds__(1024) void k_voxel_blend_mips(MipArgs a) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int B = a.brick, res = a.res, sl = a.slab_log2, bl = a.brick_levels;
  const int nx = res >> sl, nb = res >> bl;
  const int bx = static_cast<int>(blockIdx.x) % nx, by = (static_cast<int>(blockIdx.x) / nx) % nb,
            bz = static_cast<int>(blockIdx.x) / (nx * nb);
  const int tid = static_cast<int>(threadIdx.x), threads = static_cast<int>(blockDim.x);
  const uint32_t corner = static_cast<uint32_t>(((bz << bl) * res + (by << bl)) * res + (bx << sl));
  // Level 0: voxelblend.comp:8-18.  With 16^3 bricks a thread blends 16 texels
  // (one load of target and volume each).
  if (B == kBrick) {
    const int r = tid >> (sl - 4), x = (tid & ((1 << (sl - 4)) - 1)) << 4, y = r & 15, z = r >> 4;
    const uint32_t g = corner + static_cast<uint32_t>((z * res + y) * res + x);
    const uint4 tr = *reinterpret_cast<const uint4*>(a.target + g);
    const uint4 orow = *reinterpret_cast<const uint4*>(a.mips + g);
    uint4 nr = make_uint4(0u, 0u, 0u, 0u);
    if ((tr.x | tr.y | tr.z | tr.w | orow.x | orow.y | orow.z | orow.w) != 0u) {
      const uint32_t tw[4] = {tr.x, tr.y, tr.z, tr.w}, ow[4] = {orow.x, orow.y, orow.z, orow.w};
      uint32_t nw[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t packed = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          packed |= static_cast<uint32_t>(blend_voxel((tw[k] >> (8 * b)) & 0xffu, (ow[k] >> (8 * b)) & 0xffu, a.f))
                    << (8 * b);
        nw[k] = packed;
      }
      nr = make_uint4(nw[0], nw[1], nw[2], nw[3]);
      if (((nr.x ^ orow.x) | (nr.y ^ orow.y) | (nr.z ^ orow.z) | (nr.w ^ orow.w)) != 0u)
        *reinterpret_cast<uint4*>(a.mips + g) = nr;
    }
    *reinterpret_cast<uint4*>(lds + tid * 16) = nr;
  } else {
    for (int t = tid; t < B * B * B; t += threads) {
      const int x = t & (B - 1), y = (t >> bl) & (B - 1), z = t >> (2 * bl);
      const uint32_t g = corner + static_cast<uint32_t>((z * res + y) * res + x);
      const uint8_t q = blend_voxel(a.target[g], a.mips[g], a.f);
      a.mips[g] = q;
      lds[t] = q;
    }
  }
  __syncthreads();
  // Levels 1..log2(B) inside the slab: voxelmipmap.comp:8-12.
  int src = 0, dst = 1 << (sl + 2 * bl);
  for (int k = 1; k <= bl; ++k) {
    const int lx = sl - k, ly = bl - k, wk = res >> k, n = 1 << (lx + 2 * ly);
    uint8_t* out = a.mips + a.mip_offset[k];
    for (int t = tid; t < n; t += threads) {
      const int x = t & ((1 << lx) - 1), y = (t >> lx) & ((1 << ly) - 1), z = t >> (lx + ly);
      // The children: pairs along x of two rows of two slices.
      const uint8_t* c = lds + src + ((((2 * z) << (ly + 1)) + 2 * y) << (lx + 1)) + 2 * x;
      const int row = 2 << lx, slice = row << (ly + 1);
      const uint32_t p0 = *reinterpret_cast<const uint16_t*>(c), p1 = *reinterpret_cast<const uint16_t*>(c + row);
      const uint32_t p2 = *reinterpret_cast<const uint16_t*>(c + slice),
                     p3 = *reinterpret_cast<const uint16_t*>(c + slice + row);
      const uint32_t sum = (p0 & 0xffu) + (p1 & 0xffu) + (p2 & 0xffu) + (p3 & 0xffu) + (p0 >> 8) + (p1 >> 8) +
                           (p2 >> 8) + (p3 >> 8);
      const uint8_t q = static_cast<uint8_t>((sum + 4u) >> 3);
      lds[dst + t] = q;
      out[static_cast<uint32_t>((((bz << ly) + z) * wk + ((by << ly) + y)) * wk + (bx << lx) + x)] = q;
    }
    __syncthreads();
    src = dst;
    dst += n;
  }
}

struct CornerArgs {
  uint8_t* mips;
  VoxelCorner* corners;
  uint32_t mip_offset[16];
  uint32_t corner_offset[17];
  uint32_t run_offset[17];  // runs of 64 corners before level l
  int res;
  int levels;
  int brick, brick_levels;   // levels 0..brick_levels come from the brick kernel
};

// Corner (rx, ry, rz) of a level of w texels: the footprint of the texels at
// (rx - 1, ry - 1, rz - 1) and one up, clamped to the edge, as the trilinear
// polynomial's coefficients.
__device__ __forceinline__ VoxelCorner corner_of(const uint8_t* lvl, int w, int rx, int ry, int rz) {
  const int x0 = max(rx - 1, 0), x1 = min(rx, w - 1);
  const int y0 = max(ry - 1, 0) * w, y1 = min(ry, w - 1) * w;
  const int z0 = max(rz - 1, 0) * w * w, z1 = min(rz, w - 1) * w * w;
  const uint32_t row[4] = {static_cast<uint32_t>(z0 + y0), static_cast<uint32_t>(z0 + y1),
                           static_cast<uint32_t>(z1 + y0), static_cast<uint32_t>(z1 + y1)};  // y bit | z bit << 1
  // Per row: A = t at x, B = t at x + 1 minus t at x.  The record's words are
  // (A, B) of row 0, then their differences in y, in z and in y and z; all
  // are whole and below 2048, exact in FP32 and FP16.
  float A[4], B[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    A[r] = static_cast<float>(lvl[row[r] + static_cast<uint32_t>(x0)]);
    B[r] = static_cast<float>(lvl[row[r] + static_cast<uint32_t>(x1)]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) B[r] = B[r] - A[r];
  const float lo[4] = {A[0], A[1] - A[0], A[2] - A[0], (A[3] - A[2]) - (A[1] - A[0])};
  const float hi[4] = {B[0], B[1] - B[0], B[2] - B[0], (B[3] - B[2]) - (B[1] - B[0])};
  VoxelCorner c;
#pragma unroll
  for (int r = 0; r < 4; ++r) c.row[r] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo[r], hi[r]));
  return c;
}

// The corner-expanded copy of every level, and the levels above the brick
// size (more than one brick per axis).  Workgroup 0 builds those upper
// levels from level brick_levels in LDS (voxelmipmap.comp:8-12), stores
// them and expands their corners from LDS; the other workgroups expand the
// levels the brick kernel wrote.  (The kernel boundary after the brick
// kernel makes every brick's writes visible; an in-kernel device-scope fence
// per brick costs an L2 write-back on this multi-XCD part.)
// Dynamic LDS: (res / B)^3 + (res / 2B)^3 + ... bytes when upper levels exist.
//
// A wave expands runs of 64 corners, neighbours along x, so that its eight
// texel loads and the 16-byte store are each contiguous over the lanes (four
// corners of a row in each lane kept the address unit busy: 256^3, 287 MB
// written, 115 us; 66 us with the runs, bound by the writes; 128^3: 19 and 12 us).
__global__ __launch_bounds__(256) void k_voxel_corners(CornerArgs a) {
  extern __shared__ uint8_t up[];
  const int top = a.brick_levels + 1;  // first upper level
  if (blockIdx.x == 0) {
    if (top >= a.levels) return;
    const int nb = a.res / a.brick;
    const int tid = static_cast<int>(threadIdx.x);
    const uint8_t* lb = a.mips + a.mip_offset[a.brick_levels];
    for (int t = tid; t < nb * nb * nb; t += 256) up[t] = lb[t];
    __syncthreads();
    int usrc = 0, udst = nb * nb * nb;
    for (int k = top; k < a.levels; ++k) {
      const int wp = a.res >> (k - 1), wk = a.res >> k, lk = a.levels - 1 - k;  // wk = 2^lk
      uint8_t* out = a.mips + a.mip_offset[k];
      for (int t = tid; t < wk * wk * wk; t += 256) {
        const uint8_t q = mean8(up + usrc, wp, t & (wk - 1), (t >> lk) & (wk - 1), t >> (2 * lk));
        up[udst + t] = q;
        out[t] = q;
      }
      __syncthreads();
      const uint32_t c = static_cast<uint32_t>(wk) + 1u, n = c * c * c;
      for (uint32_t i = tid; i < n; i += 256u)
        a.corners[a.corner_offset[k] + i] = corner_of(up + udst, wk, static_cast<int>(i % c),
                                                      static_cast<int>(i / c % c), static_cast<int>(i / (c * c)));
      usrc = udst;
      udst += wk * wk * wk;
    }
    return;
  }
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x - 1u) * 4u + (threadIdx.x >> 6));
  const uint32_t total = a.run_offset[min(top, a.levels)];
  int l = 0;
  for (uint32_t r = wave; r < total; r += (gridDim.x - 1u) * 4u) {
    while (l + 1 < a.levels && r >= a.run_offset[l + 1]) ++l;
    const int w = a.res >> l;
    const uint32_t c = static_cast<uint32_t>(w) + 1u, i0 = (r - a.run_offset[l]) * 64u, i = i0 + lane;
    uint32_t x, y, z;
    if (c >= 64u) {  // at most one row ends in the run
      const uint32_t row = i0 / c;
      z = row / c;
      y = row - z * c;
      x = i - row * c;
      if (x >= c) {
        x -= c;
        ++y;
      }
      if (y >= c) {
        y = 0u;
        ++z;
      }
    } else {
      const uint32_t row = i / c;
      x = i - row * c;
      z = row / c;
      y = row - z * c;
    }
    if (i >= c * c * c) continue;
    a.corners[a.corner_offset[l] + static_cast<size_t>(i)] =
        corner_of(a.mips + a.mip_offset[l], w, static_cast<int>(x), static_cast<int>(y), static_cast<int>(z));
  }
}

}  // namespace

void launch_voxelize(const drv_volume& vol, int res, const float* positions, const uint32_t* indices, uint32_t n_tri,
                     const float* world, uint8_t* target, hipStream_t s) {
  if (n_tri == 0) return;
  VoxelizeArgs a;
  for (int i = 0; i < 3; ++i) {
    a.vmin[i] = vol.volume_world_min[i];
    a.vmax[i] = vol.volume_world_max[i];
  }
  for (int i = 0; i < 16; ++i) a.world[i] = world[i];
  a.positions = positions;
  a.indices = indices;
  a.n_tri = n_tri;
  a.res = res;
  a.target = target;
  a.lanes_log2 = 0;
  while (a.lanes_log2 < kVoxelizeShareLog2 && (static_cast<uint64_t>(n_tri) << (a.lanes_log2 + 1)) <= kVoxelizeLanes)
    ++a.lanes_log2;
  const uint64_t lanes = static_cast<uint64_t>(n_tri) << a.lanes_log2;
  hipLaunchKernelGGL(k_voxelize, dim3(static_cast<unsigned>((lanes + 255) / 256)), dim3(256), 0, s, a);
}

void launch_voxel_blend_mips(const VoxelLayout& L, const uint8_t* target, uint8_t* mips, float adaption,
                             hipStream_t s) {
  MipArgs a;
  a.target = target;
  a.mips = mips;
  for (int l = 0; l < L.levels && l < 16; ++l) a.mip_offset[l] = static_cast<uint32_t>(L.mip_offset[l]);
  a.res = L.res;
  a.levels = L.levels;
  a.brick = std::min(kBrick, L.res);
  int bl = 0;
  while ((1 << (bl + 1)) <= a.brick) ++bl;
  a.brick_levels = bl;
  a.f = adaption;
  // Slabs of 16 texels below 128, 32 at 128, 64 above: a workgroup for each CU.
  a.slab_log2 = L.res < 128 ? bl : L.res < 256 ? 5 : 6;
  const size_t slab = static_cast<size_t>(a.brick) * a.brick << a.slab_log2;
  size_t lds = 0;
  for (int k = 0; k <= bl; ++k) lds += slab >> (3 * k);
  const size_t texels = static_cast<size_t>(L.res) * L.res * L.res;
  const unsigned threads = a.brick == kBrick ? static_cast<unsigned>(slab / 16) : 256u;
  hipLaunchKernelGGL(k_voxel_blend_mips, dim3(static_cast<unsigned>(texels / slab)), dim3(threads), lds, s, a);
}

void launch_voxel_corners(const VoxelLayout& L, uint8_t* mips, VoxelCorner* corners, hipStream_t s) {
  CornerArgs a;
  a.mips = mips;
  a.corners = corners;
  a.res = L.res;
  a.levels = L.levels;
  a.brick = std::min(kBrick, L.res);
  int bl = 0;
  while ((1 << (bl + 1)) <= a.brick) ++bl;
  a.brick_levels = bl;
  for (int l = 0; l < L.levels; ++l) {
    a.mip_offset[l] = static_cast<uint32_t>(L.mip_offset[l]);
    a.corner_offset[l] = static_cast<uint32_t>(L.corner_offset[l]);
  }
  a.corner_offset[L.levels] = static_cast<uint32_t>(L.corner_count);
  uint32_t runs = 0;
  for (int l = 0; l < L.levels; ++l) {
    a.run_offset[l] = runs;
    const uint32_t c = static_cast<uint32_t>(L.res >> l) + 1u;
    runs += (c * c * c + 63u) / 64u;
  }
  a.run_offset[L.levels] = runs;
  const uint32_t brick_runs = a.run_offset[std::min(bl + 1, L.levels)];
  size_t upper = 0;
  if (bl + 1 < L.levels)
    for (int w = L.res / a.brick; w >= 1; w /= 2) upper += static_cast<size_t>(w) * w * w;
  // Workgroup 0 for the upper levels, the rest for the brick levels.
  const unsigned blocks = 1u + static_cast<unsigned>(std::min<size_t>((brick_runs + 3) / 4, 8192));
  hipLaunchKernelGGL(k_voxel_corners, dim3(blocks), dim3(256), upper, s, a);
}

}  // namespace drvk
