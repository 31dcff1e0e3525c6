// Object-space light cache of the EBS and DOS renderers (gfx950): the march that reads
// it and its buffer.  The cache kernels themselves live with their techniques
// (k_ebs.hip: k_lc_ebs, k_dos.hip: k_lc_dos).
//
// PreIlluminationStructuredVolume (cppvolrend/utils/preillumination.cpp:7-80) keeps a
// 2-channel (occlusion, shadow) volume, 32^3 by default, rebuilt every Update() when
// active (ebsrenderer.cpp:127-134, dosrcrenderer.cpp:134-143).  The frame is then marched
// by _common_shaders/obj_ray_marching.comp:223-333: every opaque sample reads the cache
// with GL_LINEAR / CLAMP_TO_EDGE at tex_pos / VolumeScaledSizes and shades
// rgb <- (rgb*Iocc*ka + rgb*Isdw*kd) / (ka + kd), or with Phong shading on
// (rgb*Iocc*ka + Isdw*rgb*kd*max(0, n.l)) / (ka + kd) + Isdw*ks*specular*max(0, h.n)^n
// (:186-211; a sample whose gradient vanishes keeps its colour).  Here the
// cache is fp32 (the reference stores RG16F), laid out x fastest as float2; at the
// default size it is 256 KiB and stays in L2, so its 8 taps per sample are cache hits.
// Rays as in the plain march, 16 lanes of a wavefront to each (256^3 at 1024^2 194 -> 119 us, at
// 640 x 480 375 -> 84 us; with the samples of a wavefront's rays lit 64 at a time from a queue in
// LDS the first took 270).
#include "cvr_ctx.hpp"
#include "cvr_queue.hpp"
#include <type_traits>

namespace cvr {

constexpr int kMaxLightCacheRes = 512;
template <class T> struct LcVox { typedef T type; };

// GL_LINEAR of the cache at texel coordinates p * tex_mul - 1/2 (clamped to the edge).
__device__ __forceinline__ float2 lc_sample(const float2* __restrict__ lc, int rx, int ry, int rz, const float tm[3],
                                            f3 p) {
  int x0, x1, y0, y1, z0, z1;
  float fx, fy, fz;
  lin_axis(p.x * tm[0] - 0.5f, rx, x0, x1, fx);
  lin_axis(p.y * tm[1] - 0.5f, ry, y0, y1, fy);
  lin_axis(p.z * tm[2] - 0.5f, rz, z0, z1, fz);
  const size_t sy = size_t(rx), sz = size_t(rx) * size_t(ry);
  const size_t b00 = size_t(y0) * sy + size_t(z0) * sz, b10 = size_t(y1) * sy + size_t(z0) * sz;
  const size_t b01 = size_t(y0) * sy + size_t(z1) * sz, b11 = size_t(y1) * sy + size_t(z1) * sz;
  const float2 c000 = lc[b00 + x0], c100 = lc[b00 + x1], c010 = lc[b10 + x0], c110 = lc[b10 + x1];
  const float2 c001 = lc[b01 + x0], c101 = lc[b01 + x1], c011 = lc[b11 + x0], c111 = lc[b11 + x1];
  auto lerp2 = [](float2 a, float2 b, float t) { return make_float2(a.x + t * (b.x - a.x), a.y + t * (b.y - a.y)); };
  const float2 c0 = lerp2(lerp2(c000, c100, fx), lerp2(c010, c110, fx), fy);
  const float2 c1 = lerp2(lerp2(c001, c101, fx), lerp2(c011, c111, fx), fy);
  return lerp2(c0, c1, fz);
}

struct LcK {
  int rx, ry, rz;
  float tex_mul[3];  // cache texels per world unit: res / G
  float ka, kd;      // 0 for a term that is off
  float ks;          // Phong specular weight, 0 without shadows (Kspecular counts with ApplyShadow)
};

// kMode: kGroups or kLanes, + kPhong (with Blinn-Phong).
template <typename T, int kMode>
__global__ __launch_bounds__(256) void k_lc_render(RayFrame rf, VolGeom g, LcK L, const float2* __restrict__ lc,
                                                   const float4* __restrict__ tf, int ntf, float step, float et,
                                                   PhongK ph, const float4* __restrict__ grad, QueueShape qs,
                                                   float4* __restrict__ out, unsigned long long* __restrict__ counters) {
  __shared__ RayList<kListRays> list;
  extern __shared__ float4 s_tf[];
  stage_tf_padded(s_tf, tf, ntf);
  __syncthreads();
  const float inv_k = 1.0f / (L.ka + L.kd);
  unsigned int nsamp = 0, nshade = 0;
  const f3 eye = ld3(rf.eye);
  auto lit = [&](f3 p) {
    const float2 I = lc_sample(lc, L.rx, L.ry, L.rz, L.tex_mul, p);
    if (!(kMode & kPhong)) return Lit{inv_k * (I.x * L.ka + I.y * L.kd), 0.f};
    float dd, sp;
    if (!phong_terms(grad, g, ph, p, eye, dd, sp)) return Lit{1.f, 0.f};
    return Lit{inv_k * (I.x * L.ka + I.y * (L.kd * dd)), I.y * (L.ks * sp)};
  };
  if constexpr ((kMode & kLanes) != 0) {
    int px, py;
    lane_pixel(rf, qs.first, px, py);
    lane_march<T, true, (kMode & kPhong) != 0>(rf, g, s_tf, ntf, step, et, px, py, ph.spec, out, nsamp, nshade, lit);
  } else {
    plain_march<T, true, (kMode & kPhong) != 0>(rf, g, s_tf, ntf, step, et, FramePixels(rf, qs, queue_unit<4>(qs), 4),
                                          ph.spec, list, out, nsamp, nshade, lit);
  }
  if (counters) {
    count_add(counters, 0, nsamp);
    count_add(counters, 1, nshade);
  }
}

int lc_prepare(cvr_ctx* c, const int res[3]) {
  for (int i = 0; i < 3; ++i)
    if (res[i] < 1 || res[i] > kMaxLightCacheRes) {
      set_error("light cache: light_cache_res must be in [1, 512] per axis");
      return CVR_ERR_INVALID;
    }
  const size_t n = size_t(res[0]) * size_t(res[1]) * size_t(res[2]);
  if (n > c->lc_cap) {
    if (c->d_lc) CVR_HIP_CHECK(hipFree(c->d_lc));
    c->d_lc = nullptr;
    c->lc_cap = 0;
    CVR_HIP_CHECK(device_alloc(&c->d_lc, n * sizeof(float2)));
    c->lc_cap = n;
  }
  for (int i = 0; i < 3; ++i) c->lc_res[i] = res[i];
  c->lc_valid = false;
  return CVR_OK;
}

int launch_lc_render(cvr_ctx* c, const RayFrame& rf, int apply_occ, int apply_sdw, float ka, float kd, float step,
                     float et, const PhongK& ph, float* out, hipStream_t st) {
  LcK L{};
  const VolGeom g = geom_of(c);
  L.rx = c->lc_res[0];
  L.ry = c->lc_res[1];
  L.rz = c->lc_res[2];
  const int res[3] = {L.rx, L.ry, L.rz};
  for (int i = 0; i < 3; ++i) L.tex_mul[i] = float(double(res[i]) / double(g.G[i]));
  L.ka = apply_occ ? ka : 0.f;
  L.kd = apply_sdw ? kd : 0.f;
  L.ks = apply_sdw ? ph.ks : 0.f;
  const MarchShape ms = march_shape(rf, g, step, et, ph.on, kLaneCacheRays);
  const size_t shm = size_t(c->tf_size + 2) * sizeof(float4);
  if (c->tf_size > 4096) {
    set_error("cvr_render: light-cache march: transfer function larger than 4096 entries (staged in LDS)");
    return -4;
  }
  unsigned long long* cnt = c->collect_stats ? c->d_counters : nullptr;
  auto by_mode = [&](auto t) {
    using T = typename decltype(t)::type;
    with_mode(ms.mode, [&](auto m) {
      for_launches(ms.qs, ms.blocks, 256, [&](const QueueShape& qs, int blocks) {
        hipLaunchKernelGGL((k_lc_render<T, decltype(m)::value>), dim3(blocks), dim3(256), shm, st, rf, g, L, c->d_lc,
                           c->d_tf_rgbt, c->tf_size, step, et, ph, c->d_grad, qs, reinterpret_cast<float4*>(out), cnt);
      });
    });
  };
  if (c->dtype == CVR_U8) by_mode(LcVox<uint8_t>{});
  else by_mode(LcVox<uint16_t>{});
  CVR_HIP_CHECK(hipGetLastError());
  c->lc_valid = true;
  return CVR_OK;
}

}  // namespace cvr
