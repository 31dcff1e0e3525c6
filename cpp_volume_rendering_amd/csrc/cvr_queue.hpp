// The shaded march shared by the cone tracer, DOS, EBS, the ground truth and the surrogate:
// a wavefront marches one ray at a time, 64 consecutive samples per step, and shades the
// opaque samples it meets 64 at a time.
//
// What bounds a shaded frame is the lighting of its opaque samples (tens to thousands of
// reads each), and a ray has from none to more than a thousand of them.  With one ray per
// lane, a wavefront ran as long as its longest ray, most of its lanes idle behind it, and
// the last wavefronts ran alone: on the 256^3 frames at 1024^2 the chip held 1.2 (cone
// tracer), 1.0 (DOS) and 0.3 (EBS) wavefronts per SIMD on average, of 4, 2 and 1 that fit.
// A sample's position and opacity do not depend on the lighting, so here the march runs
// ahead of it:
//  - lane k takes sample 64 n + k of the ray; the opacity recurrence runs in order through
//    the lanes (each lane from its left neighbour), so the samples taken, their opacities
//    and the early exit are those of a one-lane march, bit for bit;
//  - opaque samples go to a queue in LDS; whenever it holds 64, every lane shades one and
//    adds it to its pixel's colour in LDS.  A wavefront's rays share the queue, so all of
//    its lanes shade until its last batch.
// A wavefront's rays lie far apart in the image: neighbours are alike, and a wavefront of
// long rays would end last.
#pragma once
#include "cvr_common.hpp"

namespace cvr {

// Sample j of a ray: s = j step, segment [s, s + h], h = min(step, D - s).  The rounding
// of each operation is spelled out so that every kernel takes the same samples.
struct RaySample {
  float s, h;
};
__device__ __forceinline__ RaySample ray_sample(int j, float step, float D) {
#pragma clang fp contract(off)
  RaySample r;
  r.s = float(j) * step;
  r.h = fminf(step, D - r.s);
  return r;
}
__device__ __forceinline__ f3 ray_sample_pos(RaySample r, f3 tp, f3 dir) {
  const float t = __builtin_fmaf(0.5f, r.h, r.s);
  return mk3(__builtin_fmaf(dir.x, t, tp.x), __builtin_fmaf(dir.y, t, tp.y), __builtin_fmaf(dir.z, t, tp.z));
}

// Lighting of a sample: its colour is rgb * m + specular * s.
struct Lit {
  float m, s;
};

constexpr int kQueueCap = 128;  // a step adds at most 64 to fewer than 64 waiting
struct WaveQueue {
  float4 a[kQueueCap];  // position, compositing weight
  float4 b[kQueueCap];  // weight * rgb, ray (bits)
  float4 dir[64];       // camera-ray direction of each of the wavefront's rays
  float acc[64][4];     // and its accumulated colour
};

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// Lane k - 1's value; `first` in lane 0.
__device__ __forceinline__ float left_lane(float v, float first) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}
// Opacity after each lane's sample: w_k = w_(k-1) + (1 - w_(k-1)) alpha_k, w_(-1) = w.
// Every round makes one more lane final; three instructions each.
__device__ __forceinline__ float opacity_scan(float alpha, float w) {
  float v = w;
#pragma unroll
  for (int k = 0; k < 64; ++k) {
    const float b = left_lane(v, w);
    v = __builtin_fmaf(1.0f - b, alpha, b);
  }
  return v;
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pixel i of the image in 16 x 16 tiles, row-major, of 2 x 2 pixel groups; false past the
// image's edges.  After xcd_remap, the 64 workgroups an XCD takes in turn are one tile (the
// 256^3 cone-traced frame at 1024^2: 90 ms, 117 ms in rows of 8 x 8 tiles).
__device__ __forceinline__ bool tiled_pixel(const RayFrame& rf, int i, int& px, int& py) {
  const int tiles_x = (rf.W + 15) >> 4, t = i >> 8;
  px = (t % tiles_x) * 16 + ((i >> 1) & 14) + (i & 1);
  py = (t / tiles_x) * 16 + ((i >> 4) & 14) + ((i >> 1) & 1);
  return px < rf.W && py < rf.H;
}
inline int tiled_pixels(const RayFrame& rf) { return ((rf.W + 15) / 16) * ((rf.H + 15) / 16) * 256; }

// Rays per wavefront and workgroups (of `waves` wavefronts) of a frame: at most `most` rays (a
// power of two up to 64) while that leaves `min_waves` wavefronts.  More rays leave fewer
// part-filled last batches, fewer rays more wavefronts to even out; where the two lines lie
// is each renderer's, measured over frame sizes.
struct QueueShape {
  int rays, blocks;
};
inline QueueShape queue_shape(const RayFrame& rf, int most, int min_waves, int waves = 4) {
  const int n = tiled_pixels(rf);
  int rays = 1;
  while (rays < most && n / (rays * 2) >= min_waves) rays *= 2;
  return QueueShape{rays, (n / rays + waves - 1) / waves};
}

// Marches rays gw, gw + nw, gw + 2 nw, ... (`rays` of them, at most 64) of the frame and
// writes their pixels; gw: this wavefront's number, nw: all wavefronts.  shade(p, dir) lights
// one sample (in texture space) for each active lane; spec: specular colour of Lit::s.
template <typename T, class Shade>
__device__ __forceinline__ void queue_march(const RayFrame& rf, const VolGeom& g, const float4* s_tf, int ntf,
                                            float step, float et, int gw, int nw, int rays, const float* spec,
                                            WaveQueue& Q, float4* __restrict__ out, unsigned int& nsamp,
                                            unsigned int& nshade, Shade&& shade) {
  typedef typename VolOct<T>::type RT;
  const int lane = threadIdx.x & 63;
  // lane r sets up the wavefront's ray r
  int px = 0, py = 0;
  const bool inside = lane < rays && tiled_pixel(rf, gw + lane * nw, px, py);
  float D_r = 0.f, w_r = 0.f;
  f3 tp_r = mk3(0.f, 0.f, 0.f), dir_r = tp_r;
  bool hit = false;
  if (inside) {
    const f3 eye = ld3(rf.eye);
    dir_r = camera_ray(rf, px, py);
    float tn, tf_;
    hit = ray_box(eye, dir_r, g.G, tn, tf_);
    D_r = fabsf(tf_ - tn);
    tp_r = mk3(__builtin_fmaf(dir_r.x, tn, eye.x), __builtin_fmaf(dir_r.y, tn, eye.y),
               __builtin_fmaf(dir_r.z, tn, eye.z));
    tp_r = tp_r + mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
    Q.dir[lane] = make_float4(dir_r.x, dir_r.y, dir_r.z, 0.f);
    Q.acc[lane][0] = Q.acc[lane][1] = Q.acc[lane][2] = 0.f;
  }
  wave_lds_sync();
  uint64_t left = __ballot(hit);  // rays not begun
  int ray = -1, jb = 0, head = 0, count = 0;
  float w = 0.f, D = 0.f;
  f3 tp = tp_r, dir = dir_r;
  RT rec = {};
  for (;;) {
    while (count < 64) {
      if (ray < 0) {
        if (!left) break;
        ray = __builtin_ctzll(left);
        left &= left - 1;
        D = lane_value(D_r, ray);
        tp = mk3(lane_value(tp_r.x, ray), lane_value(tp_r.y, ray), lane_value(tp_r.z, ray));
        dir = mk3(lane_value(dir_r.x, ray), lane_value(dir_r.y, ray), lane_value(dir_r.z, ray));
        jb = 0;
        w = 0.f;
        rec = volume_oct_load<T>(g, ray_sample_pos(ray_sample(lane, step, D), tp, dir));
      }
      const RaySample r = ray_sample(jb + lane, step, D);
      const f3 p = ray_sample_pos(r, tp, dir);
      const float4 src = sample_tf(s_tf, ntf, volume_oct_lerp<T>(g, rec, p));
      // the next step's block, in flight under the compositing and the shading (past the
      // ray's end the position is finite and its clamped block in bounds)
      rec = volume_oct_load<T>(g, ray_sample_pos(ray_sample(jb + 64 + lane, step, D), tp, dir));
      const uint64_t valid = __ballot(r.s < D && jb + lane < kMaxSamples);
      const bool opaque = ((valid >> lane) & 1) && src.w > 0.0f;
      uint64_t taken = valid;  // the samples the ray comes to
      uint64_t m = __ballot(opaque);
      if (m) {
        const float alpha = opaque ? 1.0f - __expf(-src.w * r.h) : 0.f;
        const float wa = opacity_scan(alpha, w);
        const float mine = (1.0f - left_lane(wa, w)) * alpha;
        const uint64_t over = __ballot(wa > et);
        w = lane_value(wa, 63);
        if (over) {
          const int k = __builtin_ctzll(over);  // the ray ends with sample k
          taken &= (2ull << k) - 1ull;
          m &= (2ull << k) - 1ull;
          w = lane_value(wa, k);
          jb = kMaxSamples;
        }
        if ((m >> lane) & 1) {
          const int i = (head + count + __popcll(m & ((1ull << lane) - 1ull))) & (kQueueCap - 1);
          Q.a[i] = make_float4(p.x, p.y, p.z, mine);
          Q.b[i] = make_float4(mine * src.x, mine * src.y, mine * src.z, __int_as_float(ray));
        }
        count += __popcll(m);
      }
      nsamp += (taken >> lane) & 1;
      nshade += (m >> lane) & 1;
      jb += 64;
      if (valid != ~0ull || jb >= kMaxSamples) {
        if (lane == ray) w_r = w;
        ray = -1;
      }
    }
    if (count == 0) break;
    wave_lds_sync();
    const int n = min(count, 64);
    if (lane < n) {
      const int i = (head + lane) & (kQueueCap - 1);
      const float4 a = Q.a[i], b = Q.b[i];
      const int r = __float_as_int(b.w);
      const float4 d = Q.dir[r];
      const Lit l = shade(mk3(a.x, a.y, a.z), mk3(d.x, d.y, d.z));
      const float ws = a.w * l.s;
      atomicAdd(&Q.acc[r][0], __builtin_fmaf(b.x, l.m, spec[0] * ws));
      atomicAdd(&Q.acc[r][1], __builtin_fmaf(b.y, l.m, spec[1] * ws));
      atomicAdd(&Q.acc[r][2], __builtin_fmaf(b.z, l.m, spec[2] * ws));
    }
    head = (head + n) & (kQueueCap - 1);
    count -= n;
    wave_lds_sync();
  }
  if (inside) out[size_t(py) * rf.W + px] = make_float4(Q.acc[lane][0], Q.acc[lane][1], Q.acc[lane][2], w_r);
}

}  // namespace cvr
