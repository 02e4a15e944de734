// Indirect specular (INDIRECT_SPECULAR with DIRECT_SPECULAR_MAP_WRITE, the
// reference default, rendering/renderer.cpp:45-49): every cache keeps an
// S x S hemisphere env-map of the VAL radiance it reflects, in an
// R11G11B10F atlas with a mip chain.
//
//   k_specular_gather    cacheLightingRSM.comp:87-99, 240-243, 281-335: per
//                        (cache, VAL) the cache-local half vector picks a
//                        texel of the cache's map and the reflected radiance
//                        is added there;
//   k_specular_finalize  renderer.cpp:994-1045 (PrepareSpecularEnvmaps):
//                        shader/specularenvmap_mipmap.frag for every level,
//                        then shader/specularenvmap_fillholes.frag from the
//                        hole-fill level down to level 1.
//
// MI355X design.  Two waves own one cache at a time and keep a map each in LDS
// in FP32 (the reference read-modify-writes the R11G11B10F image once per
// VAL).  Their lanes take runs of Morton-consecutive VALs: mostly they reflect
// into the same texel, so a lane sums in registers and adds into the LDS map only
// when its texel changes (LDS float atomics to one address serialize, which made
// per-VAL adds four times slower).  With shadows in blocks of at least 16 VALs the
// runs are units of 16, and only those that light the cache: a wave tests 64 units
// at a time for shadowing and flux, queues the rest and works off the queue 64 at
// a time, so that no lane idles beside dark units (80 % of the units of a cache of
// specular_1080p).  Otherwise a lane's run is a 64th of the VALs.  The light's
// FP32 sums go to a per-cache work buffer that accumulates over the lights of a
// frame; the finalize kernel (one workgroup per cache) quantizes, builds the mips
// and fills holes in LDS and writes every level of the cache's atlas region once.
//
// Texel index S: ivec2(HemisphericalProjection(h) * S + 0.5) reaches S for
// half vectors near the horizon, so the reference's image store lands in
// the first column / row of the next cache in the atlas (or outside the
// image, where it is dropped).  The map here is (S+1) x (S+1): the extra
// column / row / corner are routed to the atlas neighbours by the finalize
// kernel, which adds them after the neighbour's own sum (the reference's
// unsynchronised read-modify-write of that texel has no defined order).
#include "drv_internal.hpp"
#include "k_common.hpp"
#include "k_specular.hpp"

namespace drvk {
namespace {

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct SpecGatherArgs {
  float cam[3];
  const float* caches;
  int stride;
  const Counter* counter;
  const float4* runs;  // VPLs by runs (launch_prepare_vpls)
  uint32_t n_vpl;
  const float* vis;  // [block][vis_pitch] or null (unshadowed)
  uint32_t vis_pitch;
  uint32_t interval;        // VPLs per shadow block, a power of two
  uint32_t interval_log2;
  int S;
  float* work;   // [cache][S * S][3]
  float* spill;  // [cache][2S + 1][3]: column x = S (y = 0..S-1), row y = S (x = 0..S-1), corner
  int first;     // 1: the first light of the cache list overwrites the work sums
};

// ivec2(p * S + 0.5) clamped to [0, S] (NaN -> 0): the clamp runs on the
// float, so the conversion is always in range.
__device__ __forceinline__ int texel_index(float p, int S) {
  const float fs = static_cast<float>(S);
  return static_cast<int>(fminf(fmaxf(__builtin_fmaf(p, fs, 0.5f), 0.0f), fs));
}

// A lane's sum over the VALs in a row that reflect into one texel.
struct TexelSum {
  int tex = -1;
  float r = 0.0f, g = 0.0f, b = 0.0f;
  __device__ __forceinline__ void flush(float* map) const {
    if (tex < 0) return;
    float* t = map + tex * 3;
    atomicAdd(t, r);
    atomicAdd(t + 1, g);
    atomicAdd(t + 2, b);
  }
};

// One VAL (position and disc area, flux, normal) of cache wp.
__device__ __forceinline__ void specular_val(TexelSum& run, float* map, int S, const f3& wp, const LocalFrame& fr,
                                             float4 vp, float4 vf, float4 vn, float shadowing) {
  // radianceIn, cacheLightingRSM.comp:246-264 (the SH gather's expressions)
  const float tx0 = vp.x - wp.x, ty0 = vp.y - wp.y, tz0 = vp.z - wp.z;
  const float d2 = __builtin_fmaf(tz0, tz0, __builtin_fmaf(ty0, ty0, tx0 * tx0));
  const float inv = __builtin_amdgcn_rsqf(d2);
  const float tx = tx0 * inv, ty = ty0 * inv, tz = tz0 * inv;
  const float nd = -__builtin_fmaf(vn.z, tz, __builtin_fmaf(vn.y, ty, vn.x * tx));
  const float f = fminf(1.0f, fmaxf(0.0f, nd)) * shadowing * __builtin_amdgcn_rcpf(d2 + vp.w);
  // cacheLightingRSM.comp:281-335
  const f3 l = to_local(fr, tx, ty, tz);
  const float hz0 = l.z + 1.0f;
  const float hi = __builtin_amdgcn_rsqf(__builtin_fmaf(hz0, hz0, __builtin_fmaf(l.y, l.y, l.x * l.x)));
  const float hx = l.x * hi, hy = l.y * hi, hz = hz0 * hi;
  float proj[2];
  hemi_projection(hx, hy, hz, proj);
  const int ix = texel_index(proj[0], S), iy = texel_index(proj[1], S);
  const float k = f * fminf(1.0f, fmaxf(0.0f, __builtin_fmaf(hz, l.z, __builtin_fmaf(hy, l.y, hx * l.x))));
  const float cr = vf.x * k, cg = vf.y * k, cb = vf.z * k;
  if (cr == 0.0f && cg == 0.0f && cb == 0.0f) return;  // changes nothing
  const int tex = iy * (S + 1) + ix;
  if (tex != run.tex) {
    run.flush(map);
    run.tex = tex;
    run.r = cr;
    run.g = cg;
    run.b = cb;
  } else {
    run.r += cr;
    run.g += cg;
    run.b += cb;
  }
}

// Dynamic LDS: 4 maps of (S+1)^2 RGB floats.  Wave half h of a cache's two takes
// the half h of the units (kQueue) or of every lane's run into its own map, and
// the pair writes map 0 + map 1 out (a fixed order), so twice as many waves, each
// half as long, balance the SIMDs.  The queue is 128 units, two in each lane's
// registers (in LDS it took a third of the waves of 32x32 maps).
template <bool kQueue>
__global__ __launch_bounds__(256) void k_specular_gather(SpecGatherArgs a) {
  extern __shared__ float lds[];
  const int S = a.S, S1 = S + 1;
  const uint32_t map_floats = static_cast<uint32_t>(S1 * S1 * 3);
  const uint32_t lane = threadIdx.x & 63u, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t pair = w >> 1, half = w & 1u;
  float* map = lds + w * map_floats;
  const float* map0 = lds + (2u * pair) * map_floats;
  const float* map1 = map0 + map_floats;
  const uint32_t live = a.counter->live;
  for (uint32_t base = blockIdx.x * 2u; base < live; base += gridDim.x * 2u) {  // workgroup-uniform
    const uint32_t c = base + pair;
    const bool active = c < live;
    for (uint32_t i = lane; i < map_floats; i += 64u) map[i] = 0.0f;
    wave_lds_sync();
    if (active) {
      const float* e = a.caches + static_cast<size_t>(c) * a.stride;
      const f3 wp = make3(e[0], e[1], e[2]);
      const LocalFrame fr = local_view_space(a.cam, wp);
      if (kQueue) {
        const uint32_t units = a.n_vpl / kVplUnit, mid = units / 2u, u1 = half ? units : mid;
        const float4 *positions = a.runs, *fluxes = a.runs + a.n_vpl, *normals = fluxes + a.n_vpl;
        uint32_t next = half ? mid : 0u, queued = 0u;
        uint32_t unit = next, more_unit = 0u;  // entries `lane` and 64 + lane of the queue
        float lit_by = 0.0f, more_lit_by = 0.0f;
        while (next < u1 || queued != 0u) {
          if (next < u1) {
            const uint32_t u = min(next + lane, u1 - 1u);
            const float sh = a.vis[static_cast<size_t>(u * kVplUnit >> a.interval_log2) * a.vis_pitch + c];
            const uint32_t flux = __float_as_uint(fluxes[u].w);
            // (Zero times an odd VAL counts.)
            const bool lit = next + lane < u1 && ((sh != 0.0f && flux != 0u) || flux == kOddFlux);
            const uint64_t m = __ballot(lit);
            const uint32_t n = static_cast<uint32_t>(__popcll(m));
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                            __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
            // Lit units go to the lanes from `queued` on, the others to the lanes left.
            const int to = static_cast<int>(4u * ((queued + (lit ? rank : n + lane - rank)) & 63u));
            const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_ds_permute(to, static_cast<int>(u)));
            const float got_by = __builtin_bit_cast(
                float, __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, sh)));
            const uint32_t place = (lane - queued) & 63u;
            if (place < n && lane >= queued) {
              unit = got;
              lit_by = got_by;
            } else if (place < n) {
              more_unit = got;
              more_lit_by = got_by;
            }
            queued += n;
            next += 64u;
            if (queued < 64u && next < u1) continue;
            if (queued == 0u) break;
          }
          if (lane < queued) {
            TexelSum run;
#pragma unroll 2
            for (uint32_t i = 0; i < kVplUnit; ++i) {
              const size_t r = static_cast<size_t>(i) * units + unit;
              specular_val(run, map, S, wp, fr, positions[r], fluxes[r], normals[r], lit_by);
            }
            run.flush(map);
          }
          queued -= min(queued, 64u);
          unit = more_unit;
          lit_by = more_lit_by;
        }
      } else {
        const uint32_t per_run = a.n_vpl / 64u, mid = per_run / 2u, i0 = half ? mid : 0u, i1 = half ? per_run : mid;
        float shadowing = 1.0f;
        TexelSum run;
        for (uint32_t i = i0; i < i1; ++i) {
          const uint32_t m = lane * per_run + i;
          const float4* r = a.runs + 3 * static_cast<size_t>(i * 64u + lane);
          const float4 vp = r[0], vf = r[1], vn = r[2];
          // The block's shadowing changes every `interval` VALs.
          if (a.vis && (i == i0 || (m & (a.interval - 1u)) == 0u))
            shadowing = a.vis[static_cast<size_t>(m >> a.interval_log2) * a.vis_pitch + c];
          specular_val(run, map, S, wp, fr, vp, vf, vn, shadowing);
        }
        run.flush(map);
      }
    }
    __syncthreads();  // both maps of every pair are complete
    if (active) {
      float* wk = a.work + static_cast<size_t>(c) * S * S * 3;
      float* sp = a.spill + static_cast<size_t>(c) * (2 * S + 1) * 3;
      for (uint32_t i = half * 64u + lane; i < map_floats; i += 128u) {
        const int tex = static_cast<int>(i / 3u), ch = static_cast<int>(i % 3u);
        const int x = tex % S1, y = tex / S1;
        const float val = map0[i] + map1[i];
        if (x < S && y < S) {
          float* o = wk + (y * S + x) * 3 + ch;
          *o = a.first ? val : *o + val;
        } else {
          const int k = (x == S && y < S) ? y : (y == S && x < S) ? S + x : 2 * S;
          sp[k * 3 + ch] = val;
        }
      }
    }
    __syncthreads();  // the maps are zeroed again for the next caches
  }
}

struct SpecFinalArgs {
  const Counter* counter;
  int S, levels, fill;
  uint32_t per_row;
  uint32_t width;
  uint64_t level_offset[kSpecMaxLevels];
  float norm;
  float* work;
  const float* spill;
  uint32_t* atlas;
};

__device__ __forceinline__ float quantize(float v, int ch) {
  const int m = ch == 2 ? 5 : 6;
  return uf_decode(uf_encode(v, m), m);
}

// Dynamic LDS: the decoded RGB texels of every level of one cache.
__global__ __launch_bounds__(256) void k_specular_finalize(SpecFinalArgs a) {
  extern __shared__ float lv[];
  const int S = a.S, SS = S * S;
  const uint32_t live = a.counter->live;
  const uint32_t N = a.per_row;
  int lofs[kSpecMaxLevels];
  {
    int o = 0;
#pragma unroll
    for (int l = 0; l < kSpecMaxLevels; ++l) {
      lofs[l] = o;
      const int sl = S >> l;
      o += sl * sl;
    }
  }
  const int tid = static_cast<int>(threadIdx.x);
  for (uint32_t c = blockIdx.x; c < live; c += gridDim.x) {
    const uint32_t cx = c % N, cy = c / N;
    const bool has_l = cx > 0u, has_u = cy > 0u;
    float* wk = a.work + static_cast<size_t>(c) * SS * 3;
    const size_t sp_stride = static_cast<size_t>(2 * S + 1) * 3;
    // Level 0: own sums plus the spill of the left, upper and upper-left
    // atlas neighbours, scaled by the base normalization, quantized.
    for (int t = tid; t < SS; t += 256) {
      const int x = t % S, y = t / S;
      float v[3] = {wk[t * 3], wk[t * 3 + 1], wk[t * 3 + 2]};
      const bool from_l = x == 0 && has_l, from_u = y == 0 && has_u;
      if (from_l) {
        const float* s = a.spill + static_cast<size_t>(c - 1u) * sp_stride + y * 3;
        for (int ch = 0; ch < 3; ++ch) v[ch] += s[ch];
      }
      if (from_u) {
        const float* s = a.spill + static_cast<size_t>(c - N) * sp_stride + (S + x) * 3;
        for (int ch = 0; ch < 3; ++ch) v[ch] += s[ch];
      }
      if (from_l && from_u) {
        const float* s = a.spill + static_cast<size_t>(c - N - 1u) * sp_stride + 2 * S * 3;
        for (int ch = 0; ch < 3; ++ch) v[ch] += s[ch];
      }
      if (from_l || from_u)
        for (int ch = 0; ch < 3; ++ch) wk[t * 3 + ch] = v[ch];
      for (int ch = 0; ch < 3; ++ch) lv[t * 3 + ch] = quantize(v[ch] * a.norm, ch);
    }
    __syncthreads();
    // specularenvmap_mipmap.frag: a bilinear tap at the centre of each
    // destination texel = mean of its 2x2 source texels.
    for (int l = 1; l < a.levels; ++l) {
      const int sl = S >> l, sp = S >> (l - 1);
      const float* src = lv + lofs[l - 1] * 3;
      float* dst = lv + lofs[l] * 3;
      for (int t = tid; t < sl * sl; t += 256) {
        const int x = t % sl, y = t / sl;
        const int i00 = ((2 * y) * sp + 2 * x) * 3, i10 = i00 + 3, i01 = i00 + sp * 3, i11 = i01 + 3;
        for (int ch = 0; ch < 3; ++ch)
          dst[t * 3 + ch] =
              quantize(((src[i00 + ch] + src[i10 + ch]) + (src[i01 + ch] + src[i11 + ch])) * 0.25f, ch);
      }
      __syncthreads();
    }
    // specularenvmap_fillholes.frag, levels fill .. 1.
    for (int i = a.fill; i >= 1; --i) {
      const int si = S >> i, sd = S >> (i - 1);
      const float* src = lv + lofs[i] * 3;
      float* dst = lv + lofs[i - 1] * 3;
      for (int t = tid; t < si * si; t += 256) {
        const int x = t % si, y = t / si;
        const float s[3] = {src[t * 3], src[t * 3 + 1], src[t * 3 + 2]};
        if ((s[0] + s[1]) + s[2] < 0.0001f) continue;  // discard
        int di[4];
        di[0] = ((2 * y) * sd + 2 * x) * 3;
        di[1] = di[0] + 3;
        di[2] = di[0] + sd * 3;
        di[3] = di[2] + 3;
        float d[4][3];
        float sum[3] = {0.0f, 0.0f, 0.0f};
        for (int k = 0; k < 4; ++k) {
          for (int ch = 0; ch < 3; ++ch) d[k][ch] = dst[di[k] + ch];
          if ((d[k][0] + d[k][1]) + d[k][2] == 0.0f)
            for (int ch = 0; ch < 3; ++ch) d[k][ch] = s[ch];
          for (int ch = 0; ch < 3; ++ch) sum[ch] += d[k][ch];
        }
        float en[3];
        for (int ch = 0; ch < 3; ++ch) en[ch] = 4.0f * s[ch] / (sum[ch] + 0.00001f);
        for (int k = 0; k < 4; ++k)
          for (int ch = 0; ch < 3; ++ch) dst[di[k] + ch] = quantize(d[k][ch] * en[ch], ch);
      }
      __syncthreads();
    }
    // Every level of the cache's atlas region.
    for (int l = 0; l < a.levels; ++l) {
      const int sl = S >> l;
      const uint64_t wl = a.width >> l;
      uint32_t* out = a.atlas + a.level_offset[l];
      const float* src = lv + lofs[l] * 3;
      for (int t = tid; t < sl * sl; t += 256) {
        const int x = t % sl, y = t / sl;
        const uint64_t px = static_cast<uint64_t>(cx) * sl + x, py = static_cast<uint64_t>(cy) * sl + y;
        out[py * wl + px] = pack_r11g11b10(src[t * 3], src[t * 3 + 1], src[t * 3 + 2]);
      }
    }
    __syncthreads();  // lv is reused by the next cache
  }
}

}  // namespace

// Units of 16 VALs in a queue where whole units can be dark and there are enough
// of them for the lanes; else runs of a 64th of the VALs.  Queue / runs, 16x16 maps:
// 16384 VALs in blocks of 16, 6352 caches 139 / 312 us (32x32 maps 222 / 461); 4096
// VALs 70 / 91, 1154 caches 30 / 31 (32x32 maps 45 / 42); 1024 VALs 50 / 38 and 19 /
// 16; 64 VALs 61 / 19.  Without shadows 329 / 308, blocks of one VAL 325 / 268 (4096
// VALs; of four 95 / 99, 1154 caches 38 / 32), as nearly all units are lit.
bool specular_queue(uint32_t n_vpl, uint32_t interval, bool shadow) {
  return shadow && interval >= kVplUnit && n_vpl >= 4096u;
}

void launch_specular(const float* cam, const float* caches, int stride, const Counter* counter, const float4* vpl_runs,
                     uint32_t n_vpl, const float* vis, uint32_t vis_pitch, uint32_t interval, const SpecAtlas& at,
                     int first, int grid, hipStream_t s) {
  SpecGatherArgs g;
  for (int i = 0; i < 3; ++i) g.cam[i] = cam[i];
  g.caches = caches;
  g.stride = stride;
  g.counter = counter;
  g.runs = vpl_runs;
  g.n_vpl = n_vpl;
  g.vis = vis;
  g.vis_pitch = vis_pitch;
  g.interval = interval;
  g.interval_log2 = static_cast<uint32_t>(__builtin_ctz(interval));
  g.S = at.S;
  g.work = at.work;
  g.spill = at.spill;
  g.first = first;
  const size_t glds = static_cast<size_t>(4) * (at.S + 1) * (at.S + 1) * 3 * sizeof(float);
  // More workgroups than fit at once (each takes two caches a round): the
  // hardware deals the last ones out as others finish.
  const auto gather = specular_queue(n_vpl, interval, vis != nullptr) ? k_specular_gather<true> : k_specular_gather<false>;
  hipLaunchKernelGGL(gather, dim3(4 * grid), dim3(256), glds, s, g);

  SpecFinalArgs f;
  f.counter = counter;
  f.S = at.S;
  f.levels = at.levels;
  f.fill = at.fill;
  f.per_row = at.per_row;
  f.width = at.width;
  for (int l = 0; l < kSpecMaxLevels; ++l) f.level_offset[l] = at.level_offset[l];
  f.norm = specular_base_normalization(at.S);
  f.work = at.work;
  f.spill = at.spill;
  f.atlas = at.atlas;
  size_t texels = 0;
  for (int l = 0; l < at.levels; ++l) texels += static_cast<size_t>(at.S >> l) * (at.S >> l);
  hipLaunchKernelGGL(k_specular_finalize, dim3(grid), dim3(256), texels * 3 * sizeof(float), s, f);
}

}  // namespace drvk
