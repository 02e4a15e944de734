// Brute-force RSM lighting: every pixel sums the light of every VAL of the
// RSM directly (shader/bruteforcersm.frag:15-88, drawn by
// Renderer::ApplyRSMsBruteForce, rendering/renderer.cpp:851-874).  It is the
// reference's own unshadowed ground truth for the cache path.
//
// A workgroup owns an 8x8 pixel tile, one lane per pixel; its four waves take
// a quarter of the VALs each and their sums are combined in LDS in a fixed
// order (a small window still fills the chip).  The VAL records are
// wave-uniform (scalar loads), four at a time: a 2x2 square of texels in
// Morton order.
//
// The kernel is bound by FP32 VALU issue, so work that cannot contribute is
// left out per group of four, and a pair costs only what depends on both the
// pixel and the VAL (the VAL's disc area comes from its record, the BRDF's
// colours multiply the sums once per pixel):
//  - groups without flux are skipped: the RSM's corners outside the light's
//    cone, 22-24 % of it;
//  - groups that face away from, or lie behind, the surface of every pixel of
//    the tile are skipped after the two cosines' signs: 59 % of the groups
//    with flux on boxes_1080p, 39 % on a 637x359 view of 300 boxes.
// 1920x1080 x 16384 VALs, diffuse: 25.6 -> 7.6 ms; 637x359 x 4096, whole BRDF:
// 1.78 -> 0.68 ms.  Two and four pixels per lane (fewer scalar loads per pair)
// took 15.8 and 16.6 ms against 14.9 ms with one, before the second skip.
#include <type_traits>

#include "drv_internal.hpp"
#include "k_common.hpp"

namespace drvk {
namespace {

struct BruteArgs {
  float inv_vp[16];
  float cam[3];
  const float* depth;
  const int16_t* normal;
  const uint8_t* albedo;
  const uint8_t* roughness_metallic;  // RG8 or null (roughness 1, metallic 0)
  const float* srgb_lut;
  const Vpl* vals;  // records of k_prepare_vpls (position, disc area, flux, normal)
  uint32_t n_vals;
  float* out;
  int width, height, accumulate;
};

// Wave-uniform reads go through the constant address space (scalar loads).
typedef float float4v __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) float4v* ValRecord;  // 3 per VAL

// The direction from a pixel to a VAL and its unnormalized cosines with the
// two normals.
struct BrutePair {
  float tx, ty, tz;
  float a, b;  // pixel normal, VAL normal (towards the pixel)
};

__device__ __forceinline__ BrutePair brute_pair(float4v pos, float4v nrm, f3 wp, f3 n) {
  BrutePair e;
  e.tx = pos.x - wp.x;
  e.ty = pos.y - wp.y;
  e.tz = pos.z - wp.z;
  e.a = __builtin_fmaf(e.tz, n.z, __builtin_fmaf(e.ty, n.y, e.tx * n.x));
  e.b = -__builtin_fmaf(nrm.z, e.tz, __builtin_fmaf(nrm.y, e.ty, nrm.x * e.tx));
  return e;
}

// One pixel.VAL pair's light, bruteforcersm.frag:58-80: s[0..2] the flux that
// arrives (diffuse term), s[3..5] the same weighted with the unnormalized
// Blinn-Phong lobe (specular term).  pos.w is the VAL's disc area, its
// distance to the light squared times the texel's solid angle
// (bruteforcersm.frag:70-73).
template <bool kDiffuseOnly>
__device__ __forceinline__ void brute_light(float* s, const BrutePair& e, float4v pos, float4v flux, f3 n, f3 c,
                                            float blinn) {
  const float dsq = __builtin_fmaf(e.tz, e.tz, __builtin_fmaf(e.ty, e.ty, e.tx * e.tx));
  if constexpr (kDiffuseOnly) {
    // The cosines' 1 / |t| each and the 1 / (|t|^2 + area) as one reciprocal;
    // selected, not clamped, so that a pixel on the VAL (|t| = 0) gets 0.
    // Both are within kFarPosition, so the product stays finite; the smallest
    // normal number added (nothing to any other product) keeps the reciprocal
    // finite.
    const float r = __builtin_amdgcn_rcpf(__builtin_fmaf(dsq, dsq + pos.w, 0x1p-126f));
    const float f = fminf(e.a, e.b) > 0.0f ? e.a * e.b * r : 0.0f;
    s[0] = __builtin_fmaf(f, flux.x, s[0]);
    s[1] = __builtin_fmaf(f, flux.y, s[1]);
    s[2] = __builtin_fmaf(f, flux.z, s[2]);
  } else {
    const float inv = __builtin_amdgcn_rsqf(dsq);
    const float tx = e.tx * inv, ty = e.ty * inv, tz = e.tz * inv;
    const float cos_theta = fminf(1.0f, fmaxf(0.0f, e.a * inv));
    const float to_int = fminf(1.0f, fmaxf(0.0f, e.b * inv));
    const float f = to_int * cos_theta * __builtin_amdgcn_rcpf(dsq + pos.w);
    // lightingfunctions.glsl:54-57: Blinn-Phong of the half vector.  The
    // exponent reaches 4000 and scales the rounding of N.H, so the sum is
    // kept in the shader's order.
    const float hx = c.x + tx, hy = c.y + ty, hz = c.z + tz;
    const float hi = __builtin_amdgcn_rsqf(__builtin_fmaf(hz, hz, __builtin_fmaf(hy, hy, hx * hx)));
    const float nh = fminf(1.0f, fmaxf(0.0f, (hx * n.x + hy * n.y + hz * n.z) * hi));
    const float fb = f * __builtin_amdgcn_exp2f(blinn * __builtin_amdgcn_logf(nh));
    s[0] = __builtin_fmaf(f, flux.x, s[0]);
    s[1] = __builtin_fmaf(f, flux.y, s[1]);
    s[2] = __builtin_fmaf(f, flux.z, s[2]);
    s[3] = __builtin_fmaf(fb, flux.x, s[3]);
    s[4] = __builtin_fmaf(fb, flux.y, s[4]);
    s[5] = __builtin_fmaf(fb, flux.z, s[5]);
  }
}

// The same in the shader's order, bruteforcersm.frag:58-80: for VALs or pixels at
// infinity or so far away that the forms above leave the range of a float.
template <bool kDiffuseOnly>
__device__ __forceinline__ void brute_far(float* s, float4v pos, float4v nrm, float4v flux, f3 wp, f3 n, f3 c,
                                          float blinn) {
  float tx = pos.x - wp.x, ty = pos.y - wp.y, tz = pos.z - wp.z;
  const float dsq = __builtin_fmaf(tz, tz, __builtin_fmaf(ty, ty, tx * tx));
  const float inv = __builtin_amdgcn_rsqf(dsq);
  tx *= inv;
  ty *= inv;
  tz *= inv;
  const float cos_theta = fminf(1.0f, fmaxf(0.0f, __builtin_fmaf(tz, n.z, __builtin_fmaf(ty, n.y, tx * n.x))));
  const float to_int = fminf(1.0f, fmaxf(0.0f, -__builtin_fmaf(nrm.z, tz, __builtin_fmaf(nrm.y, ty, nrm.x * tx))));
  const float f = to_int * cos_theta * __builtin_amdgcn_rcpf(dsq + pos.w);
  s[0] = __builtin_fmaf(f, flux.x, s[0]);
  s[1] = __builtin_fmaf(f, flux.y, s[1]);
  s[2] = __builtin_fmaf(f, flux.z, s[2]);
  if constexpr (!kDiffuseOnly) {
    const float hx = c.x + tx, hy = c.y + ty, hz = c.z + tz;
    const float hi = __builtin_amdgcn_rsqf(__builtin_fmaf(hz, hz, __builtin_fmaf(hy, hy, hx * hx)));
    const float nh = fminf(1.0f, fmaxf(0.0f, (hx * n.x + hy * n.y + hz * n.z) * hi));
    const float fb = f * __builtin_amdgcn_exp2f(blinn * __builtin_amdgcn_logf(nh));
    s[3] = __builtin_fmaf(fb, flux.x, s[3]);
    s[4] = __builtin_fmaf(fb, flux.y, s[4]);
    s[5] = __builtin_fmaf(fb, flux.z, s[5]);
  }
}

template <bool kDiffuseOnly>
__global__ __launch_bounds__(256) void k_bruteforce(BruteArgs a) {
  constexpr int kN = kDiffuseOnly ? 3 : 6;
  __shared__ float part[3][kN][64];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x * 8 + (lane & 7);
  const int y = blockIdx.y * 8 + (lane >> 3);
  const bool inside = x < a.width && y < a.height;
  const size_t p = inside ? static_cast<size_t>(y) * a.width + x : 0u;
  const float d = inside ? a.depth[p] : 0.0f;
  const bool lit = inside && d >= 0.00001f;  // background pixels (cleared depth) get no light
  // lightingfunctions.glsl:26-44: Blinn exponent
  const float rough = a.roughness_metallic ? static_cast<float>(a.roughness_metallic[2 * p]) / 255.0f : 1.0f;
  const float rsq = rough * rough;
  const float blinn = 2.0f / (rsq * rsq + 0.0005f);
  float s[kN];
#pragma unroll
  for (int k = 0; k < kN; ++k) s[k] = 0.0f;
  if (__ballot(lit) != 0ull) {
    // bruteforcersm.frag:17-28; unlit pixels (normal 0) face no VAL
    f3 wp = unproject_pixel(a.inv_vp, a.width, a.height, x, y, d);
    f3 n = unpack_normal16i(a.normal[2 * p], a.normal[2 * p + 1]);
    if (!lit) wp = n = make3(0.0f, 0.0f, 0.0f);
    f3 c = make3(a.cam[0] - wp.x, a.cam[1] - wp.y, a.cam[2] - wp.z);
    const float cl = sqrtf(c.x * c.x + c.y * c.y + c.z * c.z);
    c.x /= cl;
    c.y /= cl;
    c.z /= cl;
    // This wave's quarter of the groups of four VALs; the last wave also
    // takes the VALs after the last whole group.
    const uint32_t groups = a.n_vals / 4u;
    const uint32_t g0 = groups * w / 4u, g1 = groups * (w + 1u) / 4u;
    const ValRecord vals = (ValRecord)(a.vals);  // NOLINT(old-style-cast)
    const bool far = !(fabsf(wp.x) < kFarPosition && fabsf(wp.y) < kFarPosition && fabsf(wp.z) < kFarPosition);
    bool odd = false;
    for (uint32_t k = g0 / 16u + lane; k < (g1 + 15u) / 16u; k += 64u) odd |= __float_as_uint(a.vals[64u * k].least_cos) != 0u;
    const bool any_far = __ballot(far) != 0ull;
    // Two loops, so that the ordinary one pays nothing for the odd groups: 7.61 ms
    // without them and 7.59 with, 8.6 with both kinds in one loop (1920x1080 x
    // 16384 VALs, diffuse).
    auto sum = [&](auto with_odd) {
      for (uint32_t g = g0; g < g1; ++g) {
        const ValRecord v = vals + 12u * g;
        float4v pos[4], flux[4], nrm[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pos[j] = v[3 * j];
          flux[j] = v[3 * j + 1];
          nrm[j] = v[3 * j + 2];
        }
        const uint32_t quad_flux = __float_as_uint(flux[0].w);  // Vpl::quad_flux
        if constexpr (decltype(with_odd)::value) {
          if (any_far || quad_flux == kOddFlux) {
#pragma unroll 1
            for (int j = 0; j < 4; ++j) brute_far<kDiffuseOnly>(s, v[3 * j], v[3 * j + 2], v[3 * j + 1], wp, n, c, blinn);
            continue;
          }
        }
        if (quad_flux == 0u) continue;
        BrutePair e[4];
        float m[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          e[j] = brute_pair(pos[j], nrm[j], wp, n);
          m[j] = fminf(e[j].a, e[j].b);
        }
        if (__ballot(fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])) > 0.0f) == 0ull) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) brute_light<kDiffuseOnly>(s, e[j], pos[j], flux[j], n, c, blinn);
      }
    };
    if (__builtin_expect(!any_far && __ballot(odd) == 0ull, 1))
      sum(std::false_type());
    else
      sum(std::true_type());
    if (w == 3u)
      for (uint32_t i = 4u * groups; i < a.n_vals; ++i)
        brute_far<kDiffuseOnly>(s, vals[3u * i], vals[3u * i + 2u], vals[3u * i + 1u], wp, n, c, blinn);
  }
  if (w != 0u) {
#pragma unroll
    for (int k = 0; k < kN; ++k) part[w - 1u][k][lane] = s[k];
  }
  __syncthreads();
  if (w != 0u || !inside) return;
#pragma unroll
  for (int k = 0; k < kN; ++k) s[k] = (s[k] + part[0][k][lane]) + (part[1][k][lane] + part[2][k][lane]);
  const float metal = a.roughness_metallic ? static_cast<float>(a.roughness_metallic[2 * p + 1]) / 255.0f : 0.0f;
  const float norm = (blinn + 8.0f) / (8.0f * kPi);
  float* o = a.out + 3 * p;
  for (int k = 0; k < 3; ++k) {
    const float base = a.srgb_lut[a.albedo[3 * p + k]];
    const float diff = base + (0.02f - base) * metal;
    float v = diff * (1.0f / kPi) * s[k];
    if constexpr (!kDiffuseOnly) v = __builtin_fmaf((0.04f + (base - 0.04f) * metal) * norm, s[3 + k], v);
    v = lit ? v : 0.0f;
    o[k] = a.accumulate ? o[k] + v : v;
  }
}

}  // namespace

void launch_bruteforce(const drv_config& cfg, const drv_frame& frame, const drv_spot_light& light,
                       const drv_gbuffer& gb, const uint8_t* roughness_metallic, const float* srgb_lut,
                       const Vpl* vals, uint32_t n_vals, int diffuse_only, float* out_rgb, int accumulate,
                       hipStream_t s) {
  BruteArgs a;
  for (int i = 0; i < 16; ++i) a.inv_vp[i] = frame.inverse_view_projection[i];
  for (int i = 0; i < 3; ++i) a.cam[i] = frame.camera_position[i];
  a.depth = gb.depth;
  a.normal = gb.normal;
  a.albedo = gb.albedo;
  a.roughness_metallic = roughness_metallic;
  a.srgb_lut = srgb_lut;
  a.vals = vals;
  a.n_vals = n_vals;
  a.out = out_rgb;
  a.width = cfg.width;
  a.height = cfg.height;
  a.accumulate = accumulate;
  const dim3 grid((cfg.width + 7) / 8, (cfg.height + 7) / 8);
  if (diffuse_only)
    hipLaunchKernelGGL(k_bruteforce<true>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(k_bruteforce<false>, grid, dim3(256), 0, s, a);
}

}  // namespace drvk
