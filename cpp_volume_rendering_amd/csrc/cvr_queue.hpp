// The shaded march shared by the cone tracer, DOS, EBS, the ground truth and the surrogate:
// a wavefront marches one ray at a time, 64 consecutive samples per step (the surrogate four
// rays and 16 samples, or a lane to each of 64 rays), and shades the opaque samples it meets
// 64 at a time.  The plain and light-cache marches (plain_march, lane_march), whose samples
// are shaded by one read or none, are below.
//
// What bounds a shaded frame is the lighting of its opaque samples (tens to thousands of
// reads each), and a ray has from none to more than a thousand of them.  With one ray per
// lane, a wavefront ran as long as its longest ray, most of its lanes idle behind it, and
// the last wavefronts ran alone: on the 256^3 frames at 1024^2 the chip held 1.2 (cone
// tracer), 1.0 (DOS) and 0.3 (EBS) wavefronts per SIMD on average, of 4, 2 and 1 that fit.
// A sample's position and opacity do not depend on the lighting, so here the march runs
// ahead of it:
//  - lane k takes sample 64 n + k of the ray (of 64 samples a step); the opacity recurrence runs in order through
//    the lanes (each lane from its left neighbour), so the samples taken, their opacities
//    and the early exit are those of a one-lane march, bit for bit;
//  - opaque samples go to a queue in LDS; whenever it holds 64, every lane shades one and
//    adds it to its pixel's colour in LDS.  A wavefront's rays share the queue, so all of
//    its lanes shade until its last batch.
// A wavefront's rays lie some way apart in the image: neighbours are alike, and a wavefront of
// long rays would end last.
#pragma once
#include "cvr_common.hpp"
#include <cmath>
#include <type_traits>

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

// Opacity before each lane's sample: w_0 = w, w_(k+1) = w_k + (1 - w_k) alpha_k, in order.
// Lane k takes alpha_0 with the row shift by k, alpha_1 with that by k - 1, and so on; shifts
// that reach past its row's first lane read 0, which leaves w as it is, bit for bit.
// (In assembly: the compiler keeps the shift apart from the fused multiply-add, 3 instructions a
// round for 2.  The wait is for the shift's source, if it was written just before.)
__device__ __forceinline__ float opacity_rounds(float alpha, float w) {
#define CVR_ROUND(d)                                                                  \
  "v_sub_f32_e32 %1, 1.0, %0\n"                                                       \
  "v_fmac_f32_dpp %0, %2, %1 row_shr:" #d " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
  float t;
  asm("s_nop 1\n" CVR_ROUND(15) CVR_ROUND(14) CVR_ROUND(13) CVR_ROUND(12) CVR_ROUND(11) CVR_ROUND(10) CVR_ROUND(9)
          CVR_ROUND(8) CVR_ROUND(7) CVR_ROUND(6) CVR_ROUND(5) CVR_ROUND(4) CVR_ROUND(3) CVR_ROUND(2) CVR_ROUND(1)
      : "+v"(w), "=&v"(t)
      : "v"(alpha));
#undef CVR_ROUND
  return w;
}
__device__ __forceinline__ float opacity_after(float alpha, float w) { return __builtin_fmaf(alpha, 1.0f - w, w); }
// A whole wavefront's 64 samples: each round shifts every lane's value by one lane, and makes
// one more lane final.
__device__ __forceinline__ float left_lane(float v, float first) {  // wave_shr:1; `first` in lane 0
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), 0x138, 0xf, 0xf, false));
}
template <int kSub> __device__ __forceinline__ float opacity_before(float alpha, float w) {
  if (kSub == 1) return w;
  if (kSub == 16) return opacity_rounds(alpha, w);
  float b = w;
#pragma unroll
  for (int k = 0; k < 63; ++k) b = left_lane(opacity_after(alpha, b), w);
  return b;
}
// The last lane's value of each row of 16.
__device__ __forceinline__ float row_last(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x15f, 0xf, 0xf, true));
}

// Sum and (of values >= 0) maximum over each row of 16 lanes, in its last lane.
template <int kShift> __device__ __forceinline__ float row_shifted(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x110 + kShift, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float v) {
  v += row_shifted<1>(v);
  v += row_shifted<2>(v);
  v += row_shifted<4>(v);
  return v + row_shifted<8>(v);
}
__device__ __forceinline__ float row_max(float v) {  // as whole numbers: the same order, one instruction each
  int i = __float_as_int(v);
  i = max(i, __float_as_int(row_shifted<1>(__int_as_float(i))));
  i = max(i, __float_as_int(row_shifted<2>(__int_as_float(i))));
  i = max(i, __float_as_int(row_shifted<4>(__int_as_float(i))));
  return __int_as_float(max(i, __float_as_int(row_shifted<8>(__int_as_float(i)))));
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bits 0, 2, 4, ... 10 of v: a Z-order index's x (of v >> 1: y).
__device__ __forceinline__ int even_bits(int v) {
  v &= 0x555;
  v = (v | (v >> 1)) & 0x333;
  v = (v | (v >> 2)) & 0x70f;
  return (v | (v >> 4)) & 0x3f;
}
// Pixels of the image in square tiles of 1 << tile_log2 pixels (at most 64), row-major, each in
// Z order.
__host__ __device__ inline long long tiled_pixels(int w, int h, int tile_log2) {
  const long long m = 1 << tile_log2;
  return ((w + m - 1) / m) * ((h + m - 1) / m) * m * m;
}

// How a frame's rays are dealt out: `rays` per unit (a wavefront, or a workgroup whose four
// wavefronts share them), the tile whose pixels the units take in turn, workgroups,
// and runs of 1 << xcd_log2 workgroups per XCD (xcd_remap).  first: the launch's first workgroup of
// them (for_launches).
struct QueueShape {
  int rays, tile_log2, blocks, xcd_log2, first;
  const int* short_tiles;  // if not null, per tile of 64 x 64 pixels: this launch draws those whose entry is `want`
  int want;
};
// Tiles of 64 x 64 pixels: a unit's rays lie 32 (rays 4) or 16 (rays 16) pixels apart, so long
// and short ones mix, while the units that run at once stay together (256^3 cone-traced frame
// at 512^2: 18.7 ms, 23.7 ms in 16 x 16 tiles; EBS 5.0 and 6.6 ms; DOS 4.5 and 6.0 ms; cone tracer and
// DOS before cone_T and the rows of dos_cone).
// Narrower frames take smaller tiles, of a unit's rays at least.  xcd_px: pixels an XCD takes in a row.
inline QueueShape queue_shape(int w, int h, int rays, int parts, int xcd_px, int waves = 4) {
  const int side = w < h ? w : h;
  QueueShape q{rays, 2, 0, 0, 0, nullptr, 0};
  while (q.tile_log2 < 6 && (1 << q.tile_log2 < side || 1 << (2 * q.tile_log2) < rays)) ++q.tile_log2;
  const int per_wg = rays * waves / parts;  // pixels of a workgroup
  q.blocks = int((tiled_pixels(w, h, q.tile_log2) + per_wg - 1) / per_wg);
  while (per_wg << q.xcd_log2 < xcd_px) ++q.xcd_log2;
  return q;
}
// How the tiles of short rays of a frame of shape q are dealt out: `rays` to a wavefront.
inline QueueShape short_shape(const RayFrame& rf, const QueueShape& q, int rays) {
  QueueShape s = queue_shape(rf.W, rf.H, rays, 1, 256);
  s.short_tiles = q.short_tiles;
  s.want = 1;
  return s;
}
// A frame of 2^28 pixels takes up to 2^36 lanes (64 a pixel where four wavefronts share four rays):
// launch(shape, workgroups) for each launch of it.
template <class F> inline void for_launches(QueueShape q, int total, int threads, F&& launch) {
  for_runs(total, threads, [&](long long first, int blocks) {
    q.first = int(first);
    launch(q, blocks);
  });
}
// The unit of this wavefront.
template <int kParts> __device__ __forceinline__ int queue_unit(const QueueShape& q) {
  const int waves = int(blockDim.x) >> 6, bid = q.first + xcd_remap(blockIdx.x, gridDim.x, q.xcd_log2);
  return kParts > 1 ? bid : bid * waves + int(threadIdx.x >> 6);
}

// Whether this launch leaves the workgroup's tile to another (the units of a workgroup are of one tile).
template <int kParts> __device__ __forceinline__ bool tile_left_out(const QueueShape& q) {
  if (!q.short_tiles) return false;
  const int tile = queue_unit<kParts>(q) >> (2 * q.tile_log2 - __builtin_ctz(q.rays));
  return q.short_tiles[__builtin_amdgcn_readfirstlane(tile)] != q.want;
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// A value all 64 lanes share, in a scalar register; a group's value as it is.
template <int kSub> __device__ __forceinline__ float group_uniform(float v) {
  return kSub == 64 ? __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))) : v;
}

// The pixels of unit u of a frame: the units of a tile take its pixels in turn, `group`
// neighbours at a time (a power of two, as `rays`).
struct FramePixels {
  const RayFrame& rf;
  int x0, y0, first, stride, group;
  __device__ __forceinline__ FramePixels(const RayFrame& r, const QueueShape& q, int u, int g = 1) : rf(r), group(g) {
    const int tiles_x = (rf.W + (1 << q.tile_log2) - 1) >> q.tile_log2;
    const int log2 = 2 * q.tile_log2 - __builtin_ctz(q.rays);  // of the units of a tile
    const int t = u >> log2;
    stride = 1 << log2;
    first = (u & (stride - 1)) * g;
    x0 = (t % tiles_x) << q.tile_log2;
    y0 = (t / tiles_x) << q.tile_log2;
  }
  __device__ __forceinline__ bool operator()(int k, int& px, int& py) const {
    const int j = first + (k & ~(group - 1)) * stride + (k & (group - 1));
    px = x0 + even_bits(j);
    py = y0 + even_bits(j >> 1);
    return px < rf.W && py < rf.H;
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
  static_assert(kSub == 64 || kSub == 16 || kSub == 1, "groups are wavefronts, DPP rows or lanes");
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
          const float wb = opacity_before<kSub>(alpha, w), wa = opacity_after(alpha, wb);
          mine = (1.0f - wb) * alpha;
          // (a transparent sample ends no ray, also where the threshold is below 0)
          const uint64_t over = (__ballot(opaque && wa > et) >> base) & kGroupMask;
          const int last = over ? __builtin_ctzll(over) : kSub - 1;  // over: the ray ends with that sample
          w = kSub == 64 ? lane_value(wa, last) : kSub == 1 ? wa : __shfl(wa, base + last);
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

// sample_tf of a table with its first and last entry twice, for d in [0, 1] (a density is, to
// a rounding): the two entries lie side by side, and no index needs a clamp.
__device__ __forceinline__ float4 sample_tf_padded(const float4* tf, int ntf, float d) {
  const float x = d * float(ntf) - 0.5f, fl = floorf(x), f = x - fl;
  const float4* e = tf + int(fl);
  const float4 a = e[1], b = e[2];
  return make_float4(a.x + f * (b.x - a.x), a.y + f * (b.y - a.y), a.z + f * (b.z - a.z), a.w + f * (b.w - a.w));
}
__device__ __forceinline__ void stage_tf_padded(float4* s_tf, const float4* __restrict__ tf, int ntf) {
  for (int i = threadIdx.x; i < ntf + 2; i += blockDim.x) s_tf[i] = tf[min(max(i - 1, 0), ntf - 1)];
}

// The march whose lighting costs less than the queue: lit(p) gives the factor of the colour of
// the sample at p where it is met.  A lane adds up its own samples' colours and a group of 16 lanes
// adds up its lanes' when its ray ends.  The first wavefront sets up the workgroup's rays, one per lane;
// then all of them take rays from the list.  et is not below 0 (march_shape).
constexpr int kListRays = 32;  // of a workgroup (64: 128^3 at 512^2 60 us, 50 with 32)
template <int kRays> struct RayList {
  float4 tp[kRays];   // entry point (texture space), length
  float4 dir[kRays];  // direction, pixel (bits)
  int count, next;    // rays listed, taken
};
template <typename T, bool kPadded, bool kSpec, class Pix, class Lit1>
__device__ __forceinline__ void plain_march(const RayFrame& rf, const VolGeom& g, const float4* tfp, int ntf,
                                            float step, float et, Pix&& pix, const float* spec, RayList<kListRays>& Q,
                                            float4* __restrict__ out, unsigned int& nsamp, unsigned int& nshade,
                                            Lit1&& lit) {
  constexpr int kSub = 16;
  const int lane = threadIdx.x & 63, sub = lane % kSub, base = lane - sub;
  const uint64_t below_group = (1ull << base) - 1ull;
  if (threadIdx.x < 64) {
    int px = 0, py = 0;
    const bool inside = lane < kListRays && pix(lane, px, py);
    bool hit = false;
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f), d = t;
    if (inside) {
      const f3 eye = ld3(rf.eye), r = camera_ray(rf, px, py);
      float tn, tf_;
      hit = ray_box(eye, r, g.G, tn, tf_);
      f3 e = mk3(__builtin_fmaf(r.x, tn, eye.x), __builtin_fmaf(r.y, tn, eye.y), __builtin_fmaf(r.z, tn, eye.z));
      e = e + mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
      t = make_float4(e.x, e.y, e.z, fabsf(tf_ - tn));
      d = make_float4(r.x, r.y, r.z, __int_as_float(py * rf.W + px));
      if (!hit) out[py * rf.W + px] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const uint64_t hits = __ballot(hit);
    if (hit) {
      const int slot = __popcll(hits & ((1ull << lane) - 1ull));
      Q.tp[slot] = t;
      Q.dir[slot] = d;
    }
    if (lane == 0) {
      Q.count = __popcll(hits);
      Q.next = 0;
    }
  }
  __syncthreads();
  const int nhit = __builtin_amdgcn_readfirstlane(Q.count);
  f3 tp, dir;
  float4 acc;  // this lane's share of the colour; opacity of the ray
  float D;
  int jb, pixel;
  bool live = false;  // the group has a ray
  // the next rays for the groups without one (none left: D below every s)
  auto take = [&]() {
    const uint64_t need = __ballot(!live && sub == 0);
    int next = 0;
    if (lane == 0) next = atomicAdd(&Q.next, __popcll(need));
    next = __builtin_amdgcn_readfirstlane(next);
    if (!live) {
      const int mine = next + __popcll(need & below_group), i = min(mine, kListRays - 1);
      const float4 a = Q.tp[i], b = Q.dir[i];
      live = mine < nhit;
      tp = live ? mk3(a.x, a.y, a.z) : mk3(0.f, 0.f, 0.f);
      dir = live ? mk3(b.x, b.y, b.z) : mk3(0.f, 0.f, 0.f);
      D = live ? a.w : -1.f;
      pixel = __float_as_int(b.w);
      jb = sub;
      acc = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto load = [&](RaySample& s, VolTap<T>& v) {
    s = ray_sample(jb, step, D);
    v = volume_tap_load<T>(g, ray_sample_pos(s, tp, dir));
  };
  take();
  if (!__any(live)) return;
  // One step; the next step's blocks are in flight under it.  False: no rays left.
  auto go = [&](const RaySample& r, const VolTap<T>& tap, RaySample& r1, VolTap<T>& tap1) {
    const bool in_range = jb < kMaxSamples;
    jb += kSub;
    load(r1, tap1);
    const float d = volume_tap_lerp<T>(tap);
    const float4 src = kPadded ? sample_tf_padded(tfp, ntf, d) : sample_tf(tfp, ntf, d);
    const bool valid = r.s < D && in_range;
    const bool opaque = valid && src.w > 0.0f;
    const float alpha = opaque ? 1.0f - __expf(-src.w * r.h) : 0.f;
    const uint64_t valids = __ballot(valid);
    const float w0 = acc.w;
    float wa = w0;
    uint64_t over = 0;
    bool taken = valid;
    if (__any(opaque)) {
      const float wb = opacity_before<kSub>(alpha, acc.w);
      wa = opacity_after(alpha, wb);
      over = __ballot(wa > et);
      // the ray ends with the first sample over: those after it are not taken
      taken = valid && !(wb > et);
      float mine = taken ? (1.0f - wb) * alpha : 0.f;
      if (opaque && taken) {
        const Lit l = lit(ray_sample_pos(r, tp, dir));
        if (kSpec) {
          const float ws = mine * l.s;
          acc.x = __builtin_fmaf(spec[0], ws, acc.x);
          acc.y = __builtin_fmaf(spec[1], ws, acc.y);
          acc.z = __builtin_fmaf(spec[2], ws, acc.z);
        }
        mine *= l.m;
      }
      // others' colours may be anything (a transparent entry's NaN): 0 x NaN is NaN.  (Added up above instead, the
      // 16-bit light-cache march takes 73 registers, 72 here: 64^3 at 300^2 51.5 us, 45.8.)
      const bool on = opaque && taken;
      acc.x = on ? __builtin_fmaf(mine, src.x, acc.x) : acc.x;
      acc.y = on ? __builtin_fmaf(mine, src.y, acc.y) : acc.y;
      acc.z = on ? __builtin_fmaf(mine, src.z, acc.z) : acc.z;
      acc.w = row_last(wa);
      nshade += opaque && taken;
    }
    nsamp += taken;
    if (over | ~valids) {
      // some group's ray has ended (or some group has none)
      const unsigned int mine = (unsigned int)(over >> base) & 0xffffu;
      const bool ended = mine != 0 || !((valids >> (base + kSub - 1)) & 1);
      if (__any(ended && live)) {
        // the opacity does not fall along a ray: that of its last sample is the largest
        const float4 c = make_float4(row_sum(acc.x), row_sum(acc.y), row_sum(acc.z), row_max(taken ? wa : w0));
        if (ended && live && sub == kSub - 1) out[pixel] = c;
        if (ended) live = false;
        take();
        if (!__any(live)) return false;
        if (ended) load(r1, tap1);
      }
    }
    return true;
  };
  RaySample ra, rb;
  VolTap<T> ta, tb;
  load(ra, ta);
  while (go(ra, ta, rb, tb) && go(rb, tb, ra, ta)) {
  }
}

// The same march with a lane to a ray, for frames whose rays are alike: no samples are taken past a
// ray's end, and the opacity recurrence needs no other lane.  Samples in groups of four, the next
// group's blocks in flight under one (two register sets alternate).
template <typename T, bool kPadded, bool kSpec, class Lit1>
__device__ __forceinline__ void lane_march(const RayFrame& rf, const VolGeom& g, const float4* tfp, int ntf, float step,
                                           float et, int px, int py, const float* spec, float4* __restrict__ out, unsigned int& nsamp,
                                           unsigned int& nshade, Lit1&& lit) {
  constexpr int kGroup = 4;
  if (px >= rf.W || py >= rf.H) return;
  const f3 eye = ld3(rf.eye), dir = camera_ray(rf, px, py);
  float tn, tf_;
  float4 dst = make_float4(0.f, 0.f, 0.f, 0.f);
  if (ray_box(eye, dir, g.G, tn, tf_)) {
    f3 tp = mk3(__builtin_fmaf(dir.x, tn, eye.x), __builtin_fmaf(dir.y, tn, eye.y), __builtin_fmaf(dir.z, tn, eye.z));
    tp = tp + mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
    const float D = fabsf(tf_ - tn);
    auto load = [&](VolTap<T>* t, int j0) {
#pragma unroll
      for (int k = 0; k < kGroup; ++k) t[k] = volume_tap_load<T>(g, ray_sample_pos(ray_sample(j0 + k, step, D), tp, dir));
    };
    auto group = [&](const VolTap<T>* t, int j0) {  // true: the ray ends in this group
      float4 src[kGroup];
      Lit l[kGroup];
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const float d = volume_tap_lerp<T>(t[k]);
        src[k] = kPadded ? sample_tf_padded(tfp, ntf, d) : sample_tf(tfp, ntf, d);
        l[k] = Lit{1.f, 0.f};
        if (!kSpec && src[k].w > 0.0f) l[k] = lit(ray_sample_pos(ray_sample(j0 + k, step, D), tp, dir));
      }
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const RaySample r = ray_sample(j0 + k, step, D);
        if (!(r.s < D) || j0 + k >= kMaxSamples) return true;
        ++nsamp;
        if (src[k].w > 0.0f) {
          ++nshade;
          if (kSpec) l[k] = lit(ray_sample_pos(r, tp, dir));
          const float alpha = 1.0f - __expf(-src[k].w * r.h), w0 = (1.0f - dst.w) * alpha, w = w0 * l[k].m;
          if (kSpec) {
            const float ws = w0 * l[k].s;
            dst.x = __builtin_fmaf(spec[0], ws, dst.x);
            dst.y = __builtin_fmaf(spec[1], ws, dst.y);
            dst.z = __builtin_fmaf(spec[2], ws, dst.z);
          }
          dst.x = __builtin_fmaf(w, src[k].x, dst.x);
          dst.y = __builtin_fmaf(w, src[k].y, dst.y);
          dst.z = __builtin_fmaf(w, src[k].z, dst.z);
          dst.w = opacity_after(alpha, dst.w);
          if (dst.w > et) return true;
        }
      }
      return false;
    };
    VolTap<T> a[kGroup], b[kGroup];
    load(a, 0);
    for (int j0 = 0;; j0 += 2 * kGroup) {
      load(b, j0 + kGroup);
      if (group(a, j0)) break;
      load(a, j0 + 2 * kGroup);
      if (group(b, j0 + kGroup)) break;
    }
  }
  out[py * rf.W + px] = dst;
}
// Pixel of this lane in workgroups of 16 x 16 pixels (`first`: the launch's first), a wavefront 8 x 8 of
// them.
__device__ __forceinline__ void lane_pixel(const RayFrame& rf, int first, int& px, int& py) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int tx, ty;
  super_tile(first + xcd_remap(blockIdx.x, gridDim.x), (rf.W + 15) >> 4, (rf.H + 15) >> 4, 16, 32, tx, ty);
  px = tx * 16 + (w & 1) * 8 + (lane & 7);
  py = ty * 16 + (w >> 1) * 8 + (lane >> 3);
}

// The batch's work: tiles of an image in supertiles of 64, dealt to the queues in turn, each cut into kCuts
// items.
constexpr int kQueues = 8, kCuts = 4;
struct BatchShape {
  int tiles_x, tiles_y, tw_log2, span, nq, nvols;
};
// Tiles of one image in queue q.
__host__ __device__ inline int queue_tiles(const BatchShape& s, int q) {
  const int t = s.tiles_x * s.tiles_y, st = (t + 63) >> 6;  // tiles, supertiles
  if (q >= st) return 0;
  const int mine = (st - 1 - q) / s.nq + 1;
  return (st - 1) % s.nq == q ? (mine - 1) * 64 + t - (st - 1) * 64 : mine * 64;
}
// The shape of a batch of w x h images, at most `jobs` of them of one volume.  A volume's items of a queue are
// counted in 32 bits, with room for the wavefronts that find none left: where one queue would hold 2^31 items
// (64 images of 2^26 x 1) there are kQueues.
inline BatchShape batch_shape(int w, int h, int tw_log2, int span, int queues, int nvols, int jobs) {
  const int tw = 1 << tw_log2, th = (64 >> tw_log2) * span;
  BatchShape s{(w + tw - 1) / tw, (h + th - 1) / th, tw_log2, span, queues, nvols};
  if ((long long)queue_tiles(s, 0) * kCuts * jobs >= (1ll << 31) - (1 << 20)) s.nq = kQueues;
  return s;
}

// Whether ray i of 8 x 8 rays of the frame, the corners' included, hits the volume's box.
inline bool frame_ray_hits(const RayFrame& rf, const VolGeom& g, int i) {
  const float a = (float(i & 7) / 3.5f - 1.0f) * rf.tanfov * rf.aspect, b = (float(i >> 3) / 3.5f - 1.0f) * rf.tanfov;
  float lo = 0.f, hi = INFINITY;
  for (int k = 0; k < 3; ++k) {
    const float d = rf.s[k] * a + rf.u[k] * b + rf.f[k], h = 0.5f * g.G[k];
    const float x = (-h - rf.eye[k]) / d, y = (h - rf.eye[k]) / d;
    lo = std::fmax(lo, std::fmin(x, y));
    hi = std::fmin(hi, std::fmax(x, y));
  }
  return lo < hi;
}
// How many of them do; whether all do (the corners first, which miss from outside).
inline int frame_hits(const RayFrame& rf, const VolGeom& g) {
  int n = 0;
  for (int i = 0; i < 64; ++i) n += frame_ray_hits(rf, g, i);
  return n;
}
inline bool frame_all_hit(const RayFrame& rf, const VolGeom& g) {
  for (int i : {0, 7, 56, 63})
    if (!frame_ray_hits(rf, g, i)) return false;
  return frame_hits(rf, g) == 64;
}
// How the plain and the light-cache frames are marched.
enum { kGroups = 0, kPhong = 1, kLanes = 2 };  // kLanes + kPhong: both
struct MarchShape {
  int mode, blocks;
  QueueShape qs;
};
// A lane to a ray (kLanes) takes no sample past a ray's end and needs no sum over lanes, but a frame
// takes as long as its longest rays and the lanes beside them wait: it is for frames with many rays for
// the samples of the longest, and for large ones that look at nothing but the volume.  Pixels that hit
// the box over samples along its diagonal, plain march:     in groups   a lane each
//   30^3 at 1100 x 1000                           1320           63 us        48
//   64^3 at 1100 x 1000                            620           83           84
//   100^3 at 1600 x 1300                           560          167          133
//   40^3 at 800 x 700                              500           42           38
//   100^3 at 1100 x 1000                           400          103          118
//   64^3 at 700 x 600                              210           44           53
//   400 x 380 x 390 at 1000 x 900                   80          203          415
//   64^3 at 700 x 600, from near                  1390          129          120
//   40^3 at 400 x 330, from near                   700           41           44
//   dense 200^3 at 800 x 700, from near            590          113          123
//   dense 291 x 336 x 306 from inside, 576 x 442   240           53           39
//   128^3 from inside at 701 x 433                 690          175          173
//   128^3 from inside at 400 x 327                 300           89          120
// light cache (cache and march):
//   100^3 at 1100 x 1000, from near               2430          948          913
//   64^3 at 1100 x 1000                            620          238          277
// Blinn-Phong, from near:
//   43 x 27 x 35 at 2241 x 1296                  10800         1012          730
//   64^3 at 1100 x 1000                           3800          645          613
//   100^3 at 1100 x 1000                          2430          882          913
//   64^3 at 700 x 600                             1390          260          358
constexpr float kLaneRays = 500.f, kLaneCacheRays = 2000.f, kLanePhongRays = 3500.f;
constexpr size_t kLanePixels = 1 << 17;
inline MarchShape march_shape(const RayFrame& rf, const VolGeom& g, float step, float et, bool phong, float lane_rays) {
  MarchShape m;
  m.qs = queue_shape(rf.W, rf.H, kListRays, 4, 512);
  m.blocks = m.qs.blocks;
  m.mode = phong ? kPhong : kGroups;
  const size_t px = size_t(rf.W) * rf.H;
  const int hits = frame_hits(rf, g);
  const float steps = std::sqrt(g.G[0] * g.G[0] + g.G[1] * g.G[1] + g.G[2] * g.G[2]) / step;
  // plain_march ends a ray by the opacity before a sample, lane_march with an opaque one: the same but
  // where the threshold is below 0
  if (et < 0.f || (hits == 64 && px >= kLanePixels) ||
      float(px) * float(hits) / 64.f >= steps * (phong ? kLanePhongRays : lane_rays)) {
    m.mode += kLanes;
    m.blocks = ((rf.W + 15) / 16) * ((rf.H + 15) / 16);
  }
  return m;
}
template <class F> inline void with_mode(int mode, F&& f) {
  if (mode == kLanes) f(std::integral_constant<int, kLanes>{});
  else if (mode == kLanes + kPhong) f(std::integral_constant<int, kLanes + kPhong>{});
  else if (mode == kPhong) f(std::integral_constant<int, kPhong>{});
  else f(std::integral_constant<int, kGroups>{});
}

}  // namespace cvr
