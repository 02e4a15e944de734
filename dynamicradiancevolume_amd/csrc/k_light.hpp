// Device bodies of the light pass shared by the single-view kernels
// (k_gather.hip) and the batched kernels (k_batch.hip): the VPL / shadow-
// block records of one RSM texel, one (tile, split group) item of the SH
// gather and one (tile, coefficient) item of the split reduction
// (shader/cacheLightingRSM.comp:80-374).
#pragma once

#include "drv_internal.hpp"
#include "k_common.hpp"
#include "k_sample.hpp"
#include "k_sh.hpp"

namespace drvk {

struct PrepArgs {
  float inv_lvp[16];
  float light_pos[3];
  float val_area_factor;
  float sampling_offset;
  float super_val_width;
  const uint16_t* flux;
  const int16_t* normal;
  const uint16_t* dls;
  const uint16_t* dls_shadow;
  int R;         // read level width (the Morton order's x range)
  int R_shadow;  // width of the shadow level
  int H;         // read level height: R, or R / 2 for a 2:1 RSM
  int H_shadow;
  uint32_t interval;
  int block;  // B = 2^lod texels per block side
  int flux_cut;
  Vpl* vpls;
  float4* vpl_runs;  // optional copy by runs (see launch_prepare_vpls)
  uint32_t run;
  bool run_tables;
  // Optional split plan of the gather (k_plan_gather), done by the first thread.
  Counter* plan;
  uint32_t quantum, max_splits, target_items;
  ShadowBlock* blocks;
  // Optional march plans of the blocks (kMarchSteps records each) for the
  // voxel levels of vox.
  MarchStep* march;
  VoxelView vox;
};

// World position of an RSM sample at distance d from the light
// (cacheLightingRSM.comp:154-155, 175-176).
__device__ __forceinline__ f3 rsm_position(const PrepArgs& a, float s, float t, float d) {
  float clip[4];
  mat_vec(a.inv_lvp, s * 2.0f - 1.0f, t * 2.0f - 1.0f, 0.0f, 1.0f, clip);
  const float px = clip[0] / clip[3] - a.light_pos[0];
  const float py = clip[1] / clip[3] - a.light_pos[1];
  const float pz = clip[2] / clip[3] - a.light_pos[2];
  const float l = sqrtf(px * px + py * py + pz * pz);
  return make3(a.light_pos[0] + px / l * d, a.light_pos[1] + py / l * d, a.light_pos[2] + pz / l * d);
}

__device__ __forceinline__ float rg16f_texel(const uint16_t* img, int w, int h, int i, int j, int comp) {
  i = min(w - 1, max(0, i));
  j = min(h - 1, max(0, j));
  return half_to_float(img[2 * (static_cast<size_t>(j) * w + i) + comp]);
}

// Bilinear (d, d^2) of the shadow level at a block's sampling point, the
// block's first texel (x, y) plus the sampling offset
// (cacheLightingRSM.comp:171-174).
__device__ __forceinline__ void block_depth_moments(const PrepArgs& a, uint32_t x, uint32_t y, float dd[2]) {
  const float fR = static_cast<float>(a.R), fH = static_cast<float>(a.H);
  const float ss = (static_cast<float>(x) + a.sampling_offset) / fR;
  const float st = (static_cast<float>(y) + a.sampling_offset) / fH;
  const int w = a.R_shadow, h = a.H_shadow;
  const float u = ss * static_cast<float>(w) - 0.5f, vv = st * static_cast<float>(h) - 0.5f;
  const float fu = floorf(u), fv = floorf(vv);
  const int i0 = to_int(fu), j0 = to_int(fv);
  const float al = u - fu, be = vv - fv;
#pragma unroll
  for (int c = 0; c < 2; ++c)
    dd[c] = (1.0f - al) * (1.0f - be) * rg16f_texel(a.dls_shadow, w, h, i0, j0, c) +
            al * (1.0f - be) * rg16f_texel(a.dls_shadow, w, h, i0 + 1, j0, c) +
            (1.0f - al) * be * rg16f_texel(a.dls_shadow, w, h, i0, j0 + 1, c) +
            al * be * rg16f_texel(a.dls_shadow, w, h, i0 + 1, j0 + 1, c);
}

// Cone aperture of a block from its depth moments (cacheLightingRSM.comp:180-193).
__device__ __forceinline__ float block_aperture(const PrepArgs& a, const float dd[2]) {
  const float variance = dd[1] - dd[0] * dd[0];
  const float cand = sqrtf(variance) * 2.0f / dd[0];
  // GLSL max(x, y) = (x < y) ? y : x, so a NaN candidate keeps SuperValWidth.
  return (a.super_val_width < cand) ? cand : a.super_val_width;
}

// The VPL record m (and the shadow block record when m starts a block) of
// the light in `a`, n VPLs, one per lane in order.  Lanes at and past n do not call
// it, so what neighbouring lanes exchange is whole where n holds whole groups of
// them: quad_flux from n = 4 on (nothing reads it of fewer VPLs), the light
// passes' units and blocks from their least n of 64 on.
__device__ __forceinline__ void prepare_vpl(const PrepArgs& a, uint32_t m, uint32_t n) {
  uint32_t x, y;
  morton_decode(m, x, y);
  // cacheLightingRSM.comp:141-158
  const float fR = static_cast<float>(a.R), fH = static_cast<float>(a.H);
  const float s = (static_cast<float>(x) + 0.5f) / fR;
  const float t = (static_cast<float>(y) + 0.5f) / fH;
  const size_t i = static_cast<size_t>(y) * a.R + x;
  const float d = half_to_float(a.dls[2 * i]);
  const f3 p = rsm_position(a, s, t, d);
  const f3 nrm = unpack_normal16i(a.normal[2 * i], a.normal[2 * i + 1]);
  Vpl v;
  v.px = p.x;
  v.py = p.y;
  v.pz = p.z;
  v.disc_area = d * d * a.val_area_factor;
  v.fr = half_to_float(a.flux[3 * i]);
  v.fg = half_to_float(a.flux[3 * i + 1]);
  v.fb = half_to_float(a.flux[3 * i + 2]);
  // cacheLightingRSM.comp:240-243: with INDIRECT_SPECULAR a VAL whose flux
  // sums below 0.001 is skipped (`continue`); a zero flux adds nothing.
  if (a.flux_cut && (v.fr + v.fg) + v.fb < 0.001f) v.fr = v.fg = v.fb = 0.0f;
  // Whether any VPL of the aligned group of four has flux or is odd (adjacent lanes).
  const bool odd = !(fabsf(v.px) < kFarPosition && fabsf(v.py) < kFarPosition && fabsf(v.pz) < kFarPosition &&
                     fabsf(v.disc_area) < kFarArea && fabsf(v.fr) + fabsf(v.fg) + fabsf(v.fb) < kFarArea);
  uint32_t bits = odd ? kOddFlux : __float_as_uint(v.fr) | __float_as_uint(v.fg) | __float_as_uint(v.fb);
  bits |= __shfl_xor(bits, 1);
  bits |= __shfl_xor(bits, 2);
  v.quad_flux = bits;
  v.nx = nrm.x;
  v.ny = nrm.y;
  v.nz = nrm.z;
  const uint64_t any_odd = __ballot(odd);
  v.least_cos = odd ? __builtin_nanf("") : any_odd != 0ull ? -0.0f : 0.0f;
  a.vpls[m] = v;
  if (a.vpl_runs) {
    bits |= __shfl_xor(bits, 4);
    bits |= __shfl_xor(bits, 8);
    const size_t place = (m % a.run) * (n / a.run) + m / a.run;
    float4* u = a.vpl_runs + (a.run_tables ? place : 3 * place);
    const size_t next = a.run_tables ? n : 1u;
    u[0] = make_float4(v.px, v.py, v.pz, v.disc_area);
    u[next] = make_float4(v.fr, v.fg, v.fb, __uint_as_float(bits));
    u[2 * next] = make_float4(v.nx, v.ny, v.nz, 0.0f);
  }
  // Mean normal of a block's VPLs: the B x B texel square of a block is the
  // `interval` Morton-consecutive VPLs m .. m + interval - 1, i.e. adjacent
  // lanes of one wave when interval <= 64 (sum by butterfly); larger blocks
  // are summed by their first lane.
  float bsx = nrm.x, bsy = nrm.y, bsz = nrm.z;
  if (a.blocks && a.interval <= 64u) {
    for (uint32_t o = 1; o < a.interval; o <<= 1) {
      bsx += __shfl_xor(bsx, static_cast<int>(o));
      bsy += __shfl_xor(bsy, static_cast<int>(o));
      bsz += __shfl_xor(bsz, static_cast<int>(o));
    }
  }
  if (a.blocks && (m % a.interval) == 0u) {
    float dd[2];
    block_depth_moments(a, x, y, dd);
    const f3 ap = rsm_position(a, (static_cast<float>(x) + a.sampling_offset) / fR,
                               (static_cast<float>(y) + a.sampling_offset) / fH, dd[0]);
    const float rho = block_aperture(a, dd);
    float sx = bsx, sy = bsy, sz = bsz;
    if (a.interval > 64u) {
      sx = sy = sz = 0.0f;
      const int B = a.block;
      for (int dy = 0; dy < B; ++dy)
        for (int dx = 0; dx < B; ++dx) {
          const size_t t = static_cast<size_t>(y + dy) * a.R + (x + dx);
          const f3 vn = unpack_normal16i(a.normal[2 * t], a.normal[2 * t + 1]);
          sx += vn.x;
          sy += vn.y;
          sz += vn.z;
        }
    }
    const float nl = sqrtf(sx * sx + sy * sy + sz * sz);
    const float inv = nl > 0.0f ? 1.0f / nl : 0.0f;
    a.blocks[m / a.interval] = ShadowBlock{ap.x, ap.y, ap.z, rho, sx * inv, sy * inv, sz * inv, 2.0f / (1.0f - rho)};
  }
}

// Record n of the march plan of shadow block b (one thread per record,
// n_blocks x kMarchSteps of them).  The aperture is recomputed from the
// shadow level as the block's own thread computes it (the same value).
__device__ __forceinline__ void prepare_march(const PrepArgs& a, uint32_t idx) {
  const uint32_t b = idx / kMarchSteps, n = idx % kMarchSteps;
  uint32_t x, y;
  morton_decode(b * a.interval, x, y);
  float dd[2];
  block_depth_moments(a, x, y, dd);
  const float rho = block_aperture(a, dd);
  a.march[idx] = plan_march_step(a.vox, rho, 2.0f / (1.0f - rho), static_cast<int>(n));
}

// Wave-uniform VPL records through the constant address space (scalar loads).
typedef float float4v __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) float4v* VplRecord;  // 3 per VPL

// Four VPLs first .. first + 3 for the 64 caches of a wave; shadowing[k] is
// VPL k's and lit[k] holds the lanes it may reach (kUnit; otherwise the four
// share shadowing[0] and lit[0], one shadow block's).  A VPL whose front faces
// none of those lanes adds exact zeros and is skipped after the sign of its
// cosine (Vpl::least_cos: unless its flux or distance is not finite), as are four
// VPLs without flux: the RSM's texels outside the light's cone.  Of a wave's (64 caches x VPL) steps
// that its shadow blocks leave, 29 of 60 % remain on boxes_1080p, 19 of 48 % on
// boxes_1080p_dense (a step is 48 VALU instructions, the test 7); the kernel
// went from 99 to 62 and from 796 to 325 us with the item order of k_gather.
// The four records are loaded together: the empty asm keeps the loads ahead
// of the branches, so the wave waits once.
template <bool kSh2, bool kUnit>
__device__ __forceinline__ void gather_quad(ShSums& acc, const Vpl* vpls, uint32_t first, float wx, float wy,
                                            float wz, const float* shadowing, const uint64_t* lit) {
  const VplRecord r = (VplRecord)(vpls + first);  // NOLINT(old-style-cast)
  float4v p[4], f[4], n[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    p[k] = r[3 * k];
    f[k] = r[3 * k + 1];
    n[k] = r[3 * k + 2];
  }
  asm volatile("" ::"s"(p[0]), "s"(p[1]), "s"(p[2]), "s"(p[3]), "s"(f[0]), "s"(f[1]), "s"(f[2]), "s"(f[3]), "s"(n[0]),
               "s"(n[1]), "s"(n[2]), "s"(n[3]));
  if (__float_as_uint(f[0].w) == 0u) return;  // Vpl::quad_flux
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float tx = p[k].x - wx, ty = p[k].y - wy, tz = p[k].z - wz;
    const float nd = -__builtin_fmaf(n[k].z, tz, __builtin_fmaf(n[k].y, ty, n[k].x * tx));
    if ((__ballot(!(nd <= n[k].w)) & lit[kUnit ? k : 0]) != 0ull)
      sh_accumulate<kSh2>(acc, p[k].w, f[k].x, f[k].y, f[k].z, tx, ty, tz, nd, shadowing[kUnit ? k : 0]);
  }
}

// How the VPLs of a gather are shadowed: not at all, each by a block of its
// own (shadow LOD 0), or by blocks of at least four.
constexpr int kShadowNone = 0, kShadowUnits = 1, kShadowBlocks = 2;

// One (64-cache tile, group of 4 VPL splits) item of the SH gather, one
// split per wave of the 256-thread workgroup (all four waves call it with
// the same item): raw sums of the split's VPLs, combined over the four waves
// in LDS in a fixed order, one partial per group written coefficient-major,
// partial[(group * 27 + k) * partial_pitch + cache].
template <bool kSh2, int kShadow>
__device__ __forceinline__ void gather_item(const float* __restrict__ caches, int stride, uint32_t live,
                                            const Vpl* __restrict__ vpls, uint32_t n_vpl,
                                            const float* __restrict__ vis, uint32_t vis_pitch, uint32_t interval,
                                            float* __restrict__ partial, uint32_t partial_pitch, uint32_t splits,
                                            uint32_t tile, uint32_t group, float (*part)[27][64]) {
  const uint32_t chunk = n_vpl / splits;
  const uint32_t lane = threadIdx.x & 63u;
  // Wave-uniform split index (readfirstlane lets the compiler keep the item
  // loop and the VPL / block addresses in SGPRs).
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_out = kSh2 ? 27 : 12;
  const uint32_t split = group * 4u + w;
  const uint32_t cache = tile * 64u + lane;
  const bool valid = cache < live;
  const uint32_t c = valid ? cache : 0u;
  const float* e = caches + static_cast<size_t>(c) * stride;
  const float wx = e[0], wy = e[1], wz = e[2];
  // Raw sums; the SH evaluation factors are applied at write-out.
  ShSums acc;
  sh_zero(acc);
  if (split < splits) {
    const uint32_t m0 = split * chunk, m1 = m0 + chunk;
    const uint64_t all = __ballot(valid);
    if (kShadow == kShadowBlocks) {
      uint32_t blk = m0 / interval;  // the split starts on a block boundary
      // The next block's shadowing is loaded a block ahead, so the skip test
      // below does not wait for it.  One flat loop over groups of four: with
      // an inner loop per block the compiler copied the sums between the two.
      float next = vis[static_cast<size_t>(blk) * vis_pitch + c];
      float shadowing = 0.0f;
      uint64_t lit = 0ull;
      for (uint32_t m = m0; m < m1; m += 4u) {
        if ((m & (interval - 1u)) == 0u) {
          shadowing = next;
          ++blk;
          if (m + interval < m1) next = vis[static_cast<size_t>(blk) * vis_pitch + c];
          // A block that no lane of the wave sees would add only exact zeros.
          lit = __ballot(shadowing != 0.0f) & all;
          if (lit == 0ull) m += interval - 4u;
        }
        if (lit != 0ull) gather_quad<kSh2, false>(acc, vpls, m, wx, wy, wz, &shadowing, &lit);
      }
    } else {
      for (uint32_t m = m0; m < m1; m += 4u) {
        float shadowing[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        uint64_t lit[4] = {all, all, all, all};
        if (kShadow == kShadowUnits) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            shadowing[k] = vis[static_cast<size_t>(m + k) * vis_pitch + c];
            lit[k] &= __ballot(shadowing[k] != 0.0f);
          }
        }
        gather_quad<kSh2, kShadow == kShadowUnits>(acc, vpls, m, wx, wy, wz, shadowing, lit);
      }
    }
  }
  // The workgroup's four splits of the tile are combined in LDS in a fixed
  // order, (s0 + s1) + (s2 + s3), so one partial per group goes to HBM.
  if (w & 1u) {
#pragma unroll
    for (int k = 0; k < 27; ++k)
      if (k < n_out) part[w >> 1][k][lane] = acc.s[k];
  }
  __syncthreads();
  if (!(w & 1u)) {
#pragma unroll
    for (int k = 0; k < 27; ++k)
      if (k < n_out) acc.s[k] += part[w >> 1][k][lane];
  }
  __syncthreads();
  if (w == 2u) {
#pragma unroll
    for (int k = 0; k < 27; ++k)
      if (k < n_out) part[0][k][lane] = acc.s[k];
  }
  __syncthreads();
  if (w == 0u && valid) {
    // Raw sums, coefficient-major: partial[(group * 27 + k) * pitch + cache].
    float* p = partial + static_cast<size_t>(group) * 27u * partial_pitch + cache;
#pragma unroll
    for (int k = 0; k < 27; ++k)
      if (k < n_out) p[static_cast<size_t>(k) * partial_pitch] = acc.s[k] + part[0][k][lane];
  }
}

// One (64-cache tile, coefficient x channel) item of the split reduction:
// the four waves sum interleaved quarters of the `groups` partials (lane =
// cache, every load a coalesced row), the quarters are combined in a fixed
// order through LDS, and the sum (with the SH factors) is added into the
// entry (cacheLightingRSM.comp:357-373).
__device__ __forceinline__ void reduce_item(float* caches, int stride, uint32_t live, const float* partial,
                                            uint32_t partial_pitch, uint32_t groups, uint32_t tile, uint32_t jc,
                                            const drv_sh_constants& shc, float (*part)[4][64]) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const size_t split_stride = static_cast<size_t>(27u) * partial_pitch;
  const uint32_t j = jc / 3u, ch = jc % 3u;
  const uint32_t c = tile * 64u + lane;
  const uint32_t cc = c < live ? c : 0u;
  const float* p = partial + static_cast<size_t>(jc) * partial_pitch + cc;
  const float* p0 = partial + static_cast<size_t>(ch) * partial_pitch + cc;  // raw sum of rad
  float v = 0.0f, v0 = 0.0f;
#pragma unroll 8
  for (uint32_t sp = w; sp < groups; sp += 4u) {
    v += p[sp * split_stride];
    if (j == 6u) v0 += p0[sp * split_stride];
  }
  part[0][w][lane] = v;
  part[1][w][lane] = v0;
  __syncthreads();
  if (w == 0u && c < live) {
    const float s = ((part[0][0][lane] + part[0][1][lane]) + part[0][2][lane]) + part[0][3][lane];
    const float s0 = ((part[1][0][lane] + part[1][1][lane]) + part[1][2][lane]) + part[1][3][lane];
    sh_add_coefficient(caches + static_cast<size_t>(c) * stride, j, ch, s, s0, shc);
  }
}

}  // namespace drvk
