// Tiles whose rays are short, for the frames that deal rays out to wavefront queues (cvr_queue.hpp).
//
// A unit of few rays keeps long rays apart, but where rays end after a few opaque samples (a camera inside
// a dense medium) it never fills a batch of 64: small cone-traced, DOS and ground-truth frames, whose four
// wavefronts march the same four rays, took up to three times as long as a lane per ray.  One wavefront per
// tile takes the first samples of 64 rays spread over it; the tile is short if they end there, and a second launch
// draws it with 16 rays (EBS 32) to a wavefront.  From inside dense volumes, with a lane per ray, with few rays for
// all, now:
//   DOS, 41 x 53 x 53 at 250 x 215                 126 us   392    106
//   ground truth, 89 x 103 x 108 at 248 x 176      228      392    112
//   EBS, 167 x 238 x 236 at 511 x 336             5627     8175   6170
//   cone tracer, 120 x 135 x 135 at 557 x 516    14016    14283   9930
//   cone tracer, 172 x 148 x 121, long rays      47788     9000   9125 (the look-over and a launch that finds little)
#include "cvr_ctx.hpp"
#include "cvr_queue.hpp"
#include <algorithm>

namespace cvr {

template <typename T>
__global__ __launch_bounds__(64) void k_short_tiles(RayFrame rf, VolGeom g, const float4* __restrict__ tf, int ntf,
                                                    float step, float et, int limit, int* __restrict__ tiles) {
  constexpr int kGroup = 4;
  const int tiles_x = (rf.W + 63) >> 6, t = blockIdx.x, j = int(threadIdx.x) * 64 + 27;  // one in each 8 x 8
  const int px = (t % tiles_x) * 64 + even_bits(j), py = (t / tiles_x) * 64 + even_bits(j >> 1);
  const bool inside = px < rf.W && py < rf.H;
  bool hit = false, ended = true;
  if (inside) {
    const f3 eye = ld3(rf.eye), dir = camera_ray(rf, px, py);
    float tn, tf_;
    hit = ray_box(eye, dir, g.G, tn, tf_);
    if (hit) {
      f3 tp = mk3(__builtin_fmaf(dir.x, tn, eye.x), __builtin_fmaf(dir.y, tn, eye.y), __builtin_fmaf(dir.z, tn, eye.z));
      tp = tp + mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
      const float D = fabsf(tf_ - tn);
      float w = 0.f;
      ended = false;
      for (int j0 = 0; j0 < limit && !ended; j0 += kGroup) {
        VolTap<T> tap[kGroup];
#pragma unroll
        for (int k = 0; k < kGroup; ++k) tap[k] = volume_tap_load<T>(g, ray_sample_pos(ray_sample(j0 + k, step, D), tp, dir));
#pragma unroll
        for (int k = 0; k < kGroup; ++k) {
          const RaySample r = ray_sample(j0 + k, step, D);
          const float a = sample_tf(tf, ntf, volume_tap_lerp<T>(tap[k])).w;
          if (!(r.s < D)) ended = true;
          else if (a > 0.f) {
            w = opacity_after(1.0f - __expf(-a * r.h), w);
            ended = ended || w > et;
          }
        }
      }
    }
  }
  // all but a few rays end, and none misses the box
  const uint64_t in = __ballot(inside), miss = __ballot(inside && !hit), go_on = __ballot(!ended);
  if (threadIdx.x == 0) tiles[t] = in != 0 && miss == 0 && __popcll(go_on) * 16 <= __popcll(in);
}

// Frames whose rays all hit the box (from inside it or close to it) are looked over: others have tiles of
// many misses and of short and long rays beside each other.  A ray is short up to 32 samples, fewer (pixels /
// px_per_sample) in frames whose 16 rays to a wavefront would not fill the chip.  The buffer holds the tiles of
// the largest frame (2^28 pixels, either side of 64 or more and so at most doubled by its last tile: 1 MiB) from
// the first on: one that grew would be freed under a captured frame.
constexpr size_t kMaxTiles = size_t(1) << 18;
int short_tiles(cvr_ctx* c, const RayFrame& rf, float step, float et, int px_per_sample, hipStream_t st,
                const int** tiles) {
  *tiles = nullptr;
  const VolGeom g = geom_of(c);
  const size_t px = size_t(rf.W) * rf.H;
  const int limit = int(std::min(px / px_per_sample, size_t(32)) / 4 * 4);
  if (rf.W < 64 || rf.H < 64 || limit < 4 || !frame_all_hit(rf, g)) return CVR_OK;
  const size_t n = size_t((rf.W + 63) / 64) * size_t((rf.H + 63) / 64);
  if (!c->d_short) {
    if (!c->may_allocate) return CVR_OK;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusActive;
    if (hipStreamIsCapturing(st, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      return CVR_OK;  // nothing may be allocated now
    }
    if (device_alloc(&c->d_short, kMaxTiles * sizeof(int)) != hipSuccess) {
      (void)hipGetLastError();
      return CVR_OK;
    }
  }
  if (c->dtype == CVR_U8)
    hipLaunchKernelGGL(k_short_tiles<uint8_t>, dim3(unsigned(n)), dim3(64), 0, st, rf, g, c->d_tf_rgbt, c->tf_size, step,
                       et, limit, c->d_short);
  else
    hipLaunchKernelGGL(k_short_tiles<uint16_t>, dim3(unsigned(n)), dim3(64), 0, st, rf, g, c->d_tf_rgbt, c->tf_size, step,
                       et, limit, c->d_short);
  CVR_HIP_CHECK(hipGetLastError());
  *tiles = c->d_short;
  return CVR_OK;
}

}  // namespace cvr
