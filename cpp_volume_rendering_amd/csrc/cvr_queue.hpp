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
// A wavefront's rays lie some way apart in the image: neighbours are alike, and a wavefront of
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
// kRays: the most rays a wavefront takes (LDS: 4 KiB and 48 bytes a ray).
template <int kRays> struct WaveQueue {
  float4 a[kQueueCap];  // position, compositing weight
  float4 b[kQueueCap];  // weight * rgb, ray (bits)
  float4 tp[kRays];     // each of the wavefront's rays: entry point (texture space), length
  float4 dir[kRays];    // direction
  float4 acc[kRays];    // accumulated colour, opacity
};

// Lane k - 1's value within each group of kSub lanes; `first` in the group's first lane.
template <int kSub> __device__ __forceinline__ float left_lane(float v, float first) {
  constexpr int ctrl = kSub == 64 ? 0x138 : 0x111;  // wave_shr:1, row_shr:1
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), ctrl, 0xf, 0xf, false));
}
// Opacity after each lane's sample: w_k = w_(k-1) + (1 - w_(k-1)) alpha_k, w_(-1) = w.
// Every round makes one more lane of the group final; three instructions each.
template <int kSub> __device__ __forceinline__ float opacity_scan(float alpha, float w) {
  float v = w;
#pragma unroll
  for (int k = 0; k < kSub; ++k) {
    const float b = left_lane<kSub>(v, w);
    v = __builtin_fmaf(1.0f - b, alpha, b);
  }
  return v;
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pixel i of the image in square tiles of 1 << tile_log2 pixels (at most 64), row-major, each in
// Z order; false past the image's edges.
__device__ __forceinline__ bool tiled_pixel(const RayFrame& rf, int tile_log2, int i, int& px, int& py) {
  const int tiles_x = (rf.W + (1 << tile_log2) - 1) >> tile_log2, t = i >> (2 * tile_log2), j = i & ((1 << (2 * tile_log2)) - 1);
  auto even = [](int v) {  // bits 0, 2, 4, ... of v
    v &= 0x555;
    v = (v | (v >> 1)) & 0x333;
    v = (v | (v >> 2)) & 0x70f;
    return (v | (v >> 4)) & 0x3f;
  };
  px = ((t % tiles_x) << tile_log2) + even(j);
  py = ((t / tiles_x) << tile_log2) + even(j >> 1);
  return px < rf.W && py < rf.H;
}
inline int tiled_pixels(const RayFrame& rf, int tile_log2) {
  const int m = 1 << tile_log2;
  return ((rf.W + m - 1) / m) * ((rf.H + m - 1) / m) * m * m;
}

// How a frame's rays are dealt out: `rays` per unit (a wavefront, or a workgroup whose four
// wavefronts share them: parts 4), the tile whose pixels the units take in turn, workgroups,
// and runs of 1 << xcd_log2 workgroups per XCD (xcd_remap).
struct QueueShape {
  int rays, parts, tile_log2, blocks, xcd_log2;
};
// Tiles of 64 x 64 pixels: a unit's rays lie 32 (rays 4) or 16 (rays 16) pixels apart, so long
// and short ones mix, while the units that run at once stay together (256^3 cone-traced frame
// at 512^2: 18.7 ms, 23.7 ms in 16 x 16 tiles; EBS 5.0 and 6.6 ms; DOS 4.5 and 6.0 ms).
// Narrower frames take smaller tiles.  xcd_px: pixels an XCD takes in a row.
inline QueueShape queue_shape(const RayFrame& rf, int rays, int parts, int xcd_px, int waves = 4) {
  const int side = rf.W < rf.H ? rf.W : rf.H;
  QueueShape q{rays, parts, 2, 0, 0};
  while (q.tile_log2 < 6 && 1 << q.tile_log2 < side) ++q.tile_log2;
  const int per_wg = rays * waves / parts;  // pixels of a workgroup
  q.blocks = (tiled_pixels(rf, q.tile_log2) + per_wg - 1) / per_wg;
  while (per_wg << q.xcd_log2 < xcd_px) ++q.xcd_log2;
  return q;
}
// The unit of this wavefront.
template <int kParts> __device__ __forceinline__ int queue_unit(int xcd_log2) {
  const int waves = int(blockDim.x) >> 6, bid = xcd_remap(blockIdx.x, gridDim.x, xcd_log2);
  return kParts > 1 ? bid : bid * waves + int(threadIdx.x >> 6);
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// A value all 64 lanes share, in a scalar register; a group's value as it is.
template <int kSub> __device__ __forceinline__ float group_uniform(float v) {
  return kSub == 64 ? __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))) : v;
}

// The pixels of unit u of a frame: the units of a tile take its pixels in turn, `group`
// neighbours at a time.
struct FramePixels {
  const RayFrame& rf;
  int tile_log2, first, stride, group;
  __device__ __forceinline__ FramePixels(const RayFrame& r, const QueueShape& q, int u, int g = 1)
      : rf(r), tile_log2(q.tile_log2), group(g) {
    stride = (1 << (2 * q.tile_log2)) / q.rays;  // units of a tile
    first = u / stride * (1 << (2 * q.tile_log2)) + u % stride * g;
  }
  __device__ __forceinline__ bool operator()(int k, int& px, int& py) const {
    return tiled_pixel(rf, tile_log2, first + k / group * stride * group + k % group, px, py);
  }
};

// Marches `rays` rays (at most kRays <= 64), ray k that of pixel pix(k, px, py) (false: no pixel), and
// writes their pixels: 64 / kSub rays at a time, kSub samples of each per step.
// kParts > 1: that many wavefronts of a workgroup march the same rays, each shading every
// kParts-th batch, and the first adds up their colours (every wavefront of the workgroup
// makes this call once; Q: the first one's queue, the others' follow).
// shade(on, p, dir) lights one sample (in texture space) per lane; kWhole: all 64 lanes call
// it together, `on` says which have a sample; otherwise only those with one.  spec:
// specular colour of Lit::s.
template <typename T, int kSub, bool kWhole, int kParts, int kRays, class Pix, class Shade>
__device__ __forceinline__ void queue_march(const RayFrame& rf, const VolGeom& g, const float4* s_tf, int ntf,
                                            float step, float et, int rays, Pix&& pix, const float* spec,
                                            WaveQueue<kRays>* queues, float4* __restrict__ out, unsigned int& nsamp, unsigned int& nshade,
                                            Shade&& shade) {
  typedef typename VolOct<T>::type RT;
  static_assert(kSub == 64 || kSub == 16, "groups are wavefronts or DPP rows");
  constexpr uint64_t kGroupMask = kSub == 64 ? ~0ull : (1ull << (kSub & 63)) - 1ull;
  const int lane = threadIdx.x & 63, sub = lane % kSub, base = lane - sub;
  const int part = kParts > 1 ? int(threadIdx.x >> 6) % kParts : 0;
  WaveQueue<kRays>& Q = queues[part];
  const uint64_t below = (1ull << lane) - 1ull, below_group = (1ull << base) - 1ull;
  // lane k sets up ray k; the rays that hit the box are listed in order
  int px = 0, py = 0;
  const bool inside = lane < rays && pix(lane, px, py);
  bool hit = false;
  float4 tp_k = make_float4(0.f, 0.f, 0.f, 0.f), dir_k = tp_k;
  if (inside) {
    const f3 eye = ld3(rf.eye), d = camera_ray(rf, px, py);
    float tn, tf_;
    hit = ray_box(eye, d, g.G, tn, tf_);
    f3 t = mk3(__builtin_fmaf(d.x, tn, eye.x), __builtin_fmaf(d.y, tn, eye.y), __builtin_fmaf(d.z, tn, eye.z));
    t = t + mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
    tp_k = make_float4(t.x, t.y, t.z, fabsf(tf_ - tn));
    dir_k = make_float4(d.x, d.y, d.z, 0.f);
  }
  const uint64_t hits = __ballot(hit);
  const int nhit = __popcll(hits), slot = __popcll(hits & below);
  if (hit) {
    Q.tp[slot] = tp_k;
    Q.dir[slot] = dir_k;
    Q.acc[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  wave_lds_sync();
  f3 tp = mk3(0.f, 0.f, 0.f), dir = tp;
  float D = 0.f;
  int ray = -1, jb = 0;                  // the group's ray and next sample
  int next = 0, head = 0, count = 0, batch = 0;  // next ray, queue: the same in every lane
  float w = 0.f;
  RT rec = {};
  // a new ray for the groups without one, and the blocks of every group's next samples: in
  // flight under the queue and the shading (past a ray's end the position is finite and its
  // clamped block in bounds)
  auto advance = [&]() {
    const uint64_t need = __ballot(ray < 0 && sub == 0);
    if (need && next < nhit) {
      const int mine = next + __popcll(need & below_group);
      if (ray < 0 && mine < nhit) {
        ray = mine;
        const float4 t = Q.tp[mine], d = Q.dir[mine];
        tp = mk3(group_uniform<kSub>(t.x), group_uniform<kSub>(t.y), group_uniform<kSub>(t.z));
        dir = mk3(group_uniform<kSub>(d.x), group_uniform<kSub>(d.y), group_uniform<kSub>(d.z));
        D = group_uniform<kSub>(t.w);
        jb = 0;
        w = 0.f;
      }
      next = min(nhit, next + __popcll(need));
    }
    if (ray >= 0) rec = volume_oct_load<T>(g, ray_sample_pos(ray_sample(jb + sub, step, D), tp, dir));
  };
  advance();
  for (;;) {
    while (count < 64 && __any(ray >= 0)) {
      f3 p = tp;
      float4 src = make_float4(0.f, 0.f, 0.f, 0.f);
      float mine = 0.f;
      bool emit = false;
      const int emit_ray = ray;
      if (ray >= 0) {
        const RaySample r = ray_sample(jb + sub, step, D);
        p = ray_sample_pos(r, tp, dir);
        src = sample_tf(s_tf, ntf, volume_oct_lerp<T>(g, rec, p));
        const bool valid = r.s < D && jb + sub < kMaxSamples;
        const bool opaque = valid && src.w > 0.0f;
        bool taken = valid;  // the ray comes to this sample
        bool ended = !((__ballot(valid) >> (base + kSub - 1)) & 1);
        if (__any(opaque)) {
          const float alpha = opaque ? 1.0f - __expf(-src.w * r.h) : 0.f;
          const float wa = opacity_scan<kSub>(alpha, w);
          mine = (1.0f - left_lane<kSub>(wa, w)) * alpha;
          const uint64_t over = (__ballot(wa > et) >> base) & kGroupMask;
          const int last = over ? __builtin_ctzll(over) : kSub - 1;  // over: the ray ends with that sample
          w = kSub == 64 ? lane_value(wa, last) : __shfl(wa, base + last);
          taken = valid && sub <= last;
          ended = ended || over != 0;
        }
        emit = opaque && taken;
        nsamp += taken && part == 0;
        nshade += emit && part == 0;
        jb += kSub;
        if (ended || jb >= kMaxSamples) {
          if (sub == 0) Q.acc[ray].w = w;
          ray = -1;
        }
      }
      const uint64_t m = __ballot(emit);
      if (emit) {
        const int i = (head + count + __popcll(m & below)) & (kQueueCap - 1);
        Q.a[i] = make_float4(p.x, p.y, p.z, mine);
        Q.b[i] = make_float4(mine * src.x, mine * src.y, mine * src.z, __int_as_float(emit_ray));
      }
      count += __popcll(m);
      advance();
    }
    if (count == 0) break;
    wave_lds_sync();
    const int n = min(count, 64);
    const bool on = lane < n, mine = kParts == 1 || batch % kParts == part;
    ++batch;
    if (mine && (kWhole || on)) {
      const int i = (head + (on ? lane : 0)) & (kQueueCap - 1);
      const float4 a = Q.a[i], b = Q.b[i];
      const int r = __float_as_int(b.w);
      const float4 d = Q.dir[r];
      const Lit l = shade(on, mk3(a.x, a.y, a.z), mk3(d.x, d.y, d.z));
      if (on) {
        const float ws = a.w * l.s;
        atomicAdd(&Q.acc[r].x, __builtin_fmaf(b.x, l.m, spec[0] * ws));
        atomicAdd(&Q.acc[r].y, __builtin_fmaf(b.y, l.m, spec[1] * ws));
        atomicAdd(&Q.acc[r].z, __builtin_fmaf(b.z, l.m, spec[2] * ws));
      }
    }
    head = (head + n) & (kQueueCap - 1);
    count -= n;
    wave_lds_sync();
  }
  wave_lds_sync();
  if (kParts > 1) __syncthreads();
  if (inside && part == 0) {
    float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
    if (hit) {
      c = Q.acc[slot];
      for (int i = 1; i < kParts; ++i) {
        const float4 d = queues[i].acc[slot];
        c.x += d.x;
        c.y += d.y;
        c.z += d.z;
      }
    }
    out[size_t(py) * rf.W + px] = c;
  }
  if (kParts > 1) __syncthreads();  // before the queues are used again
}

}  // namespace cvr
