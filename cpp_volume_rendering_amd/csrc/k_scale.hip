// Multi-scale output (gfx950): the rendered frame resampled to the screen size, as
// RenderFrameToScreen does it (libs/vis_utils/renderoutputframe.cpp:243-535, shaders
// vis_utils/shader/renderoutputframe/*.comp).  Three modes:
//  - multisample: the frame rendered at a multiple of the screen size, read with
//    GL_LINEAR / CLAMP_TO_EDGE at each screen pixel centre (multisample_filter.comp);
//  - downscale: the same, filtered: out = s_r s_c sum_ij k((x_r - (i+1/2)/n_r) T_r)
//    k((x_c - (j+1/2)/n_c) T_c) f_ij over the kernel's support (downscaling_filter.comp),
//    then, for the cardinal kernels, their digital filter on the result;
//  - upscale: the frame rendered at a fraction of the screen size; for the cardinal
//    kernels its digital filter first (on a copy here: the reference filters the
//    rendered frame in place), then out = sum_ij k(xi_r - i) k(xi_c - j) f_ij with
//    xi = x n - 1/2 (upscaling_filter.comp).
// Kernels (box_filter.comp ... cardinalomoms_filter.comp; Nehab and Hoppe, "A fresh look
// at generalized sampling", 2014): box, hat, Catmull-Rom, Mitchell-Netravali (B = C =
// 1/3), cardinal cubic B-spline (scaled by 6) and cardinal O-MOMS3 (scaled by 5.25).
// The digital filter inverts the kernel's sampled convolution (1, a, 1) with a = 4
// (B-spline) or 3.25 (O-MOMS): forward and backward substitution of its LU factors
// L_0 = 1/(a+1), L_i = 1/(a - L_{i-1}), truncated once they settle (8 resp. 9 factors),
// as vis_utils/filters/utils.hpp:17-44 does along every row and then every column.
// texelFetch outside the frame reads 0 here (GL leaves it undefined).
#include "cvr_ctx.hpp"

#include <cmath>

namespace cvr {

__device__ __forceinline__ float cubic_piece(int k, float u, int which) {
  // which: 0 -> k0 (x in (1, 2], u = 2 - x), 1 -> k1 (x in [0, 1], u = 1 - x)
  switch (k) {
    case CVR_FILTER_CATMULL_ROM:
      return which == 0 ? ((0.5f * u - 0.5f) * u) * u : ((-1.5f * u + 2.0f) * u + 0.5f) * u;
    case CVR_FILTER_MITCHELL_NETRAVALI:
      return which == 0 ? (((7.0f / 18.0f) * u - 1.0f / 3.0f) * u) * u
                        : (((-7.0f / 6.0f) * u + 1.5f) * u + 0.5f) * u + 1.0f / 18.0f;
    case CVR_FILTER_CARDINAL_BSPLINE3:
      return which == 0 ? (u * u) * u : ((-3.0f * u + 3.0f) * u + 3.0f) * u + 1.0f;
    default:  // O-MOMS3
      return which == 0 ? ((0.875f * u) * u + 0.125f) * u : ((-2.625f * u + 2.625f) * u + 2.25f) * u + 1.0f;
  }
}

__device__ __forceinline__ float kernel_support(int k) {
  return k == CVR_FILTER_BOX ? 1.f : (k == CVR_FILTER_HAT ? 2.f : 4.f);
}

__device__ __forceinline__ float kernel_weight(int k, float x) {
  if (k == CVR_FILTER_BOX) return (x <= -0.5f || x > 0.5f) ? 0.f : 1.f;
  x = fabsf(x);
  if (k == CVR_FILTER_HAT) return x > 1.f ? 0.f : 1.f - x;
  return x > 2.f ? 0.f : (x > 1.f ? cubic_piece(k, 2.f - x, 0) : cubic_piece(k, 1.f - x, 1));
}

__device__ __forceinline__ float4 fetch(const float4* __restrict__ f, int w, int h, int c, int r) {
  if (c < 0 || r < 0 || c >= w || r >= h) return make_float4(0.f, 0.f, 0.f, 0.f);
  return f[size_t(r) * w + c];
}

__device__ __forceinline__ void acc4(float4& a, float w, float4 v) {
  a.x += w * v.x;
  a.y += w * v.y;
  a.z += w * v.z;
  a.w += w * v.w;
}

__global__ __launch_bounds__(256) void k_multisample(const float4* __restrict__ src, int sw, int sh,
                                                     float4* __restrict__ dst, int dw, int dh) {
  const int x = blockIdx.x * 16 + (threadIdx.x & 15), y = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (x >= dw || y >= dh) return;
  const float u = (float(x) + 0.5f) / float(dw) * float(sw) - 0.5f;
  const float v = (float(y) + 0.5f) / float(dh) * float(sh) - 0.5f;
  int x0, x1, y0, y1;
  float fx, fy;
  lin_axis(u, sw, x0, x1, fx);
  lin_axis(v, sh, y0, y1, fy);
  const float4 a = src[size_t(y0) * sw + x0], b = src[size_t(y0) * sw + x1];
  const float4 c = src[size_t(y1) * sw + x0], d = src[size_t(y1) * sw + x1];
  float4 o;
  o.x = (a.x + fx * (b.x - a.x)) + fy * ((c.x + fx * (d.x - c.x)) - (a.x + fx * (b.x - a.x)));
  o.y = (a.y + fx * (b.y - a.y)) + fy * ((c.y + fx * (d.y - c.y)) - (a.y + fx * (b.y - a.y)));
  o.z = (a.z + fx * (b.z - a.z)) + fy * ((c.z + fx * (d.z - c.z)) - (a.z + fx * (b.z - a.z)));
  o.w = (a.w + fx * (b.w - a.w)) + fy * ((c.w + fx * (d.w - c.w)) - (a.w + fx * (b.w - a.w)));
  dst[size_t(y) * dw + x] = o;
}

// downscaling_filter.comp:17-57.  The 16 x 16 pixels of a workgroup share 16 sets of row weights
// and 16 of column weights, kept in LDS where a set fits (kTaps: a cubic kernel at a ratio of 7, a
// box at 31); a weight per tap and pixel took more time than the taps themselves
// (1002 x 746 to 501 x 373, B-spline: 34 us, 23 now).
constexpr int kTaps = 32;
__device__ __forceinline__ float down_weight(int kern, float x, int i, int n, int d) {
  return kernel_weight(kern, (x - (float(i) + 0.5f) / float(n)) * float(d));
}
__global__ __launch_bounds__(256) void k_downscale(const float4* __restrict__ src, int sw, int sh,
                                                   float4* __restrict__ dst, int dw, int dh, int kern) {
  __shared__ float wts[2][kTaps][16];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int jc = blockIdx.x * 16 + tx, jr = blockIdx.y * 16 + ty;
  const float s_r = float(dh) / float(sh), s_c = float(dw) / float(sw);
  const float kr = 0.5f * kernel_support(kern);
  const float x_r = (float(jr) + 0.5f) / float(dh), x_c = (float(jc) + 0.5f) / float(dw);
  const int il_r = int(ceilf((x_r - kr / float(dh)) * float(sh) - 0.5f));
  const int ir_r = int(floorf((x_r + kr / float(dh)) * float(sh) - 0.5f));
  const int il_c = int(ceilf((x_c - kr / float(dw)) * float(sw) - 0.5f));
  const int ir_c = int(floorf((x_c + kr / float(dw)) * float(sw) - 0.5f));
  const int taps = min(kTaps, int(2.f * kr * fmaxf(float(sw) / float(dw), float(sh) / float(dh))) + 2);  // of a set, at most
  for (int t = ty; t < taps; t += 16) wts[1][t][tx] = down_weight(kern, x_c, il_c + t, sw, dw);
  for (int t = tx; t < taps; t += 16) wts[0][t][ty] = down_weight(kern, x_r, il_r + t, sh, dh);
  __syncthreads();
  if (jc >= dw || jr >= dh) return;
  float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
  const bool staged = ir_c - il_c < kTaps && ir_r - il_r < kTaps;
  for (int i_r = il_r; i_r <= ir_r; ++i_r) {
    const float wr = staged ? wts[0][i_r - il_r][ty] : down_weight(kern, x_r, i_r, sh, dh);
    if (staged && il_c >= 0 && ir_c < sw && unsigned(i_r) < unsigned(sh)) {  // no tap outside the frame
      const float4* row = src + size_t(i_r) * sw;
#pragma unroll 4
      for (int i_c = il_c; i_c <= ir_c; ++i_c) acc4(f, wr * wts[1][i_c - il_c][tx], row[i_c]);
      continue;
    }
    for (int i_c = il_c; i_c <= ir_c; ++i_c)
      acc4(f, wr * (staged ? wts[1][i_c - il_c][tx] : down_weight(kern, x_c, i_c, sw, dw)),
           fetch(src, sw, sh, i_c, i_r));
  }
  const float s = s_r * s_c;
  dst[size_t(jr) * dw + jc] = make_float4(f.x * s, f.y * s, f.z * s, f.w * s);
}

// upscaling_filter.comp:17-55
__global__ __launch_bounds__(256) void k_upscale(const float4* __restrict__ src, int sw, int sh,
                                                 float4* __restrict__ dst, int dw, int dh, int kern) {
  const int jc = blockIdx.x * 16 + (threadIdx.x & 15), jr = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (jc >= dw || jr >= dh) return;
  const float kr = 0.5f * kernel_support(kern);
  const float xi_r = (float(jr) + 0.5f) / float(dh) * float(sh) - 0.5f;
  const float xi_c = (float(jc) + 0.5f) / float(dw) * float(sw) - 0.5f;
  const int il_r = int(ceilf(xi_r - kr)), ir_r = int(floorf(xi_r + kr));
  const int il_c = int(ceilf(xi_c - kr)), ir_c = int(floorf(xi_c + kr));
  float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int i_r = il_r; i_r <= ir_r; ++i_r) {
    const float wr = kernel_weight(kern, xi_r - float(i_r));
    for (int i_c = il_c; i_c <= ir_c; ++i_c)
      acc4(f, wr * kernel_weight(kern, xi_c - float(i_c)), fetch(src, sw, sh, i_c, i_r));
  }
  dst[size_t(jr) * dw + jc] = f;
}

struct DigitalL {
  int m;
  float L[9], last;  // last: L[m - 1], which all further factors equal
};

// LU factors of the digital filter: L_0 = 1/(a+1), L_i = 1/(a - L_{i-1}).
static DigitalL digital_factors(int kern) {
  DigitalL d{};
  const double a = kern == CVR_FILTER_CARDINAL_BSPLINE3 ? 4.0 : 3.25;
  d.m = kern == CVR_FILTER_CARDINAL_BSPLINE3 ? 8 : 9;
  double l = 1.0 / (a + 1.0);
  for (int i = 0; i < d.m; ++i) {
    d.L[i] = float(l);
    l = 1.0 / (a - l);
  }
  d.last = d.L[d.m - 1];
  return d;
}

// linear_solve (filters/utils.hpp:17-44) of a sequence of n <= m float4 with stride `step`:
// it is first grown by reflection until it is longer than m, as there.
__device__ void solve_short(const float4* f, float4* o, int n, size_t step, const DigitalL& D) {
  const int m = D.m;
  const float Li = D.last, v_inv = Li / (1.f + Li);
  auto axpy = [](float4 a, float s, float4 b) {  // a - s*b
    return make_float4(a.x - s * b.x, a.y - s * b.y, a.z - s * b.z, a.w - s * b.w);
  };
  auto back = [](float s, float4 a, float4 b) {  // s*(a - b)
    return make_float4(s * (a.x - b.x), s * (a.y - b.y), s * (a.z - b.z), s * (a.w - b.w));
  };
  float4 g[32];  // n <= 9: reflections until longer than m (at most 2n <= 18... 4n)
  int nn = n;
  for (int i = 0; i < n; ++i) g[i] = f[i * step];
  while (nn <= m) {
    for (int i = 0; i < nn; ++i) g[nn + i] = g[nn - 1 - i];
    nn *= 2;
  }
  for (int i = 1; i < m; ++i) g[i] = axpy(g[i], D.L[i - 1], g[i - 1]);
  for (int i = m; i < nn; ++i) g[i] = axpy(g[i], Li, g[i - 1]);
  g[nn - 1] = make_float4(g[nn - 1].x * v_inv, g[nn - 1].y * v_inv, g[nn - 1].z * v_inv, g[nn - 1].w * v_inv);
  for (int i = nn - 2; i >= m - 1; --i) g[i] = back(Li, g[i], g[i + 1]);
  for (int i = m - 2; i >= 0; --i) g[i] = back(D.L[i], g[i], g[i + 1]);
  for (int i = 0; i < n; ++i) o[i * step] = g[i];
}

// One lane per sequence: nseq of them, seq_step apart, n <= m elements each.
__global__ __launch_bounds__(256) void k_digital_short(const float4* f, float4* o, int nseq, size_t seq_step, int n,
                                                       size_t step, DigitalL D) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nseq) solve_short(f + i * seq_step, o + i * seq_step, n, step, D);
}

// An affine step of a recurrence on four components, x -> a x + b.
struct Affine {
  float a;
  float4 b;
};
// The step p, then q.  The slope keeps its sign and does not reach 0: an infinity that comes
// in goes on through any number of steps as it does in a serial recurrence (0 x inf is NaN); to a
// finite value 1e-38 of it adds nothing.
__device__ __forceinline__ Affine then(const Affine& p, const Affine& q) {
  const float a = p.a * q.a;
  return {copysignf(fmaxf(fabsf(a), 1.17549435e-38f), a),
          make_float4(q.a * p.b.x + q.b.x, q.a * p.b.y + q.b.y, q.a * p.b.z + q.b.z, q.a * p.b.w + q.b.w)};
}
__device__ __forceinline__ float4 apply(const Affine& p, float4 x) {
  return make_float4(p.a * x.x + p.b.x, p.a * x.y + p.b.y, p.a * x.z + p.b.z, p.a * x.w + p.b.w);
}
__device__ __forceinline__ float4 shfl4(float4 v, int lane) {
  return make_float4(__shfl(v.x, lane), __shfl(v.y, lane), __shfl(v.z, lane), __shfl(v.w, lane));
}

// linear_solve of nseq sequences of n > m elements (element i of sequence q at
// q seq_step + i step), a wavefront for kCols sequences: each lane holds kRun successive
// elements, runs the recurrence over them from zero, and gives the affine step that its run
// makes of what comes in; a scan over the lanes gives each the value that comes into it, and the
// recurrence is run again from that.  Forward over the sequence in chunks, then back.
// Bound by the latency of the chunks' chain (load, run, scan, run): one lane per sequence
// had a chain of 2 n loads (501 x 373, B-spline: 333 us an axis; rows 10, columns 12 now).
// kCols = 1 for rows (a lane's elements fill a cache line), 4 for columns (four lanes share 64 bytes).
constexpr int kRun = 8;
template <int kCols>
__global__ __launch_bounds__(256) void k_digital(const float4* f, float4* o, int nseq, size_t seq_step, int n,
                                                 size_t step, DigitalL D) {
  constexpr int kSegs = 64 / kCols, kChunk = kSegs * kRun;
  const int lane = threadIdx.x & 63, col = lane % kCols, seg = lane / kCols;
  const int wave = (blockIdx.x * 256 + threadIdx.x) >> 6;
  if (wave * kCols >= nseq) return;  // a whole wavefront
  const int q = wave * kCols + col;
  const bool on = q < nseq;
  f += (on ? q : 0) * seq_step;
  o += (on ? q : 0) * seq_step;
  const float Li = D.last, v_inv = Li / (1.f + Li);
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 x[kRun], carry = zero;
  float L[kRun];
#pragma unroll
  for (int k = 0; k < kRun; ++k) L[k] = lane < kCols ? D.L[k] : Li;  // of this lane's run in chunk 0
  const float l7 = D.L[kRun - 1];

  // forward: x_i = f_i - c_i x_(i-1); c_0 = 0, c_i = L[i-1] up to 8, Li beyond (L[7] is Li for m = 8)
  for (int base = 0; base < n; base += kChunk) {
    const int i0 = base + seg * kRun;
    float c[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      x[k] = on && i0 + k < n ? f[size_t(i0 + k) * step] : zero;
      c[k] = base ? Li : k ? L[k - 1] : seg == 1 ? l7 : seg ? Li : 0.f;
    }
    Affine t{-c[0], x[0]};
#pragma unroll
    for (int k = 1; k < kRun; ++k) t = then(t, Affine{-c[k], x[k]});
#pragma unroll
    for (int d = 1; d < kSegs; d *= 2) {
      const int from = seg >= d ? lane - d * kCols : lane;
      const Affine p{__shfl(t.a, from), shfl4(t.b, from)};
      if (seg >= d) t = then(p, t);
    }
    // what comes into this lane's run
    const float4 out = apply(t, carry), left = shfl4(out, seg ? lane - kCols : lane);
    float4 y = carry;
    if (seg) y = left;
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      x[k] = i0 + k == 0 ? x[k]
                         : make_float4(x[k].x - c[k] * y.x, x[k].y - c[k] * y.y, x[k].z - c[k] * y.z,
                                       x[k].w - c[k] * y.w);
      y = x[k];
      if (on && i0 + k < n) o[size_t(i0 + k) * step] = x[k];
    }
    carry = shfl4(y, (kSegs - 1) * kCols + col);
  }
  // back: x_i = s_i (x_i - x_(i+1)); s_i = L[i] up to 7, Li beyond; the last is scaled by v_inv alone.
  // A lane holds the same elements as before, so it reads what it wrote itself.
  carry = zero;
  for (int base = (n - 1) / kChunk * kChunk; base >= 0; base -= kChunk) {
    const int i0 = base + seg * kRun;
    float s[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      x[k] = on && i0 + k < n ? o[size_t(i0 + k) * step] : zero;
      s[k] = base ? Li : L[k];
      if (i0 + k == n - 1) s[k] = v_inv;
    }
    auto step_of = [&](int k) {
      const float v = s[k];
      return Affine{-v, make_float4(v * x[k].x, v * x[k].y, v * x[k].z, v * x[k].w)};
    };
    Affine t = step_of(kRun - 1);
#pragma unroll
    for (int k = kRun - 2; k >= 0; --k) t = then(t, step_of(k));
#pragma unroll
    for (int d = 1; d < kSegs; d *= 2) {
      const int from = seg + d < kSegs ? lane + d * kCols : lane;
      const Affine p{__shfl(t.a, from), shfl4(t.b, from)};
      if (seg + d < kSegs) t = then(p, t);
    }
    const float4 out = apply(t, carry), right = shfl4(out, seg + 1 < kSegs ? lane + kCols : lane);
    float4 y = carry;
    if (seg + 1 < kSegs) y = right;
#pragma unroll
    for (int k = kRun - 1; k >= 0; --k) {
      const float v = s[k];
      x[k] = i0 + k >= n - 1
                 ? make_float4(v * x[k].x, v * x[k].y, v * x[k].z, v * x[k].w)
                 : make_float4(v * (x[k].x - y.x), v * (x[k].y - y.y), v * (x[k].z - y.z), v * (x[k].w - y.w));
      y = x[k];
      if (on && i0 + k < n) o[size_t(i0 + k) * step] = x[k];
    }
    carry = shfl4(y, col);
  }
}

// The filter along one axis, from f into o (which may be f).
template <int kCols>
static void digital_axis(const float4* f, float4* o, int nseq, size_t seq_step, int n, size_t step, const DigitalL& D,
                         hipStream_t st) {
  if (n <= D.m)
    hipLaunchKernelGGL(k_digital_short, dim3(unsigned((nseq + 255) / 256)), dim3(256), 0, st, f, o, nseq, seq_step, n,
                       step, D);
  else
    hipLaunchKernelGGL((k_digital<kCols>), dim3(unsigned((nseq + 4 * kCols - 1) / (4 * kCols))), dim3(256), 0, st, f,
                       o, nseq, seq_step, n, step, D);
}

// Along every row, then every column.
static void digital_filter(const float4* f, float4* o, int w, int h, int kern, hipStream_t st) {
  const DigitalL D = digital_factors(kern);
  digital_axis<1>(f, o, h, size_t(w), w, 1, D, st);
  digital_axis<4>(o, o, w, 1, h, size_t(w), D, st);
}

}  // namespace cvr

using namespace cvr;

extern "C" int cvr_multiscale_size(int screen_w, int screen_h, int mw, int mh, int* frame_w, int* frame_h) {
  if (!frame_w || !frame_h || screen_w < 1 || screen_h < 1 || mw == 0 || mh == 0) {
    set_error("cvr_multiscale_size: screen size >= 1 and nonzero multipliers required");
    return CVR_ERR_INVALID;
  }
  // UpdateScreenResolutionMultiScaling (renderoutputframe.cpp:96-112): m > 0 multiplies,
  // m < 0 divides (integer division)
  const long long w = mw > 0 ? (long long)screen_w * mw : screen_w / (-(long long)mw);
  const long long h = mh > 0 ? (long long)screen_h * mh : screen_h / (-(long long)mh);
  if (w < 1 || h < 1 || w > (1 << 16) || h > (1 << 16)) {
    set_error("cvr_multiscale_size: frame size out of range");
    return CVR_ERR_INVALID;
  }
  *frame_w = int(w);
  *frame_h = int(h);
  return CVR_OK;
}

extern "C" int cvr_resample_frame(int device, const float* src, int sw, int sh, float* dst, int dw, int dh, int mode,
                                  int kernel, float* work, void* hip_stream) {
  if (!src || !dst || sw < 1 || sh < 1 || dw < 1 || dh < 1 || sw > (1 << 16) || sh > (1 << 16) || dw > (1 << 16) ||
      dh > (1 << 16)) {
    set_error("cvr_resample_frame: device buffers and sizes in [1, 65536] required");
    return CVR_ERR_INVALID;
  }
  if (mode < CVR_SCALE_MULTISAMPLE || mode > CVR_SCALE_UPSCALE || kernel < CVR_FILTER_BOX ||
      kernel > CVR_FILTER_CARDINAL_OMOMS3) {
    set_error("cvr_resample_frame: unknown mode or kernel");
    return CVR_ERR_INVALID;
  }
  const bool cardinal = kernel == CVR_FILTER_CARDINAL_BSPLINE3 || kernel == CVR_FILTER_CARDINAL_OMOMS3;
  if (mode == CVR_SCALE_UPSCALE && cardinal && !work) {
    set_error("cvr_resample_frame: upscaling with a cardinal kernel needs a work buffer of sw*sh*4 floats");
    return CVR_ERR_INVALID;
  }
  int prev = -1;
  if (hipGetDevice(&prev) != hipSuccess) prev = -1;
  if (prev != device) CVR_HIP_CHECK(hipSetDevice(device));
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  const dim3 grid(unsigned((dw + 15) / 16), unsigned((dh + 15) / 16));
  const float4* s4 = reinterpret_cast<const float4*>(src);
  float4* d4 = reinterpret_cast<float4*>(dst);
  if (mode == CVR_SCALE_MULTISAMPLE) {
    hipLaunchKernelGGL(k_multisample, grid, dim3(256), 0, st, s4, sw, sh, d4, dw, dh);
  } else if (mode == CVR_SCALE_DOWNSCALE) {
    hipLaunchKernelGGL(k_downscale, grid, dim3(256), 0, st, s4, sw, sh, d4, dw, dh, kernel);
    if (cardinal) digital_filter(d4, d4, dw, dh, kernel, st);
  } else {
    if (cardinal) {
      float4* w4 = reinterpret_cast<float4*>(work);
      digital_filter(s4, w4, sw, sh, kernel, st);
      s4 = w4;
    }
    hipLaunchKernelGGL(k_upscale, grid, dim3(256), 0, st, s4, sw, sh, d4, dw, dh, kernel);
  }
  const hipError_t e = hipGetLastError();
  if (prev >= 0 && prev != device) (void)hipSetDevice(prev);
  if (e != hipSuccess) {
    set_error(std::string("cvr_resample_frame: ") + hipGetErrorString(e));
    return CVR_ERR_HIP;
  }
  return CVR_OK;
}
