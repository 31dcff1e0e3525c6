// Plain single-pass ray casting (front-to-back emission-absorption), gfx950.
//
// Semantics follow cppvolrend/structured/rc1pass/ray_marching_1p.comp:156-250
// (USE_TRANSPARENCY off): midpoint samples of the segment [s, s+h], h = min(step,
// D - s); the TF holds (r, g, b, extinction); alpha = 1 - exp(-ext*h); composite
// front to back; stop once accumulated alpha exceeds the threshold.
//
// With gradient shading on, every opaque sample's colour goes through ShadeBlinnPhong
// (:48-81) before it is composited: rgb*(ka + kd*max(0, n.l)) + specular*ks*
// max(0, h.n)^shininess, n the normalised GL_LINEAR gradient (samples whose gradient is
// the zero vector keep their colour).
//
// Mapping: 16 lanes take 16 successive samples of a ray, four rays per wavefront at a time
// (plain_march).  A frame's rays have from none to hundreds of samples: with a ray per lane
// a wavefront ran as long as its longest one, and a 512^2 frame gave the chip about one
// wavefront with work per SIMD, which waited for its own loads.  What bounds it now is the vector
// arithmetic of a step (about 140 instructions for 64 samples).  64^3 at 128^2 51 -> 16 us,
// 128^3 at 512^2 95 -> 50, 400 x 380 x 390 at 1000 x 900 415 -> 203; with Blinn-Phong 161 x 193 x 97
// at 1002 x 746 307 -> 168 (shaded where it is met: through the queue of the costlier renderers
// 243).  Frames of many short rays keep a lane per ray (march_shape).  The 1D transfer
// function is staged in LDS.
#include "cvr_ctx.hpp"
#include "cvr_queue.hpp"
#include <type_traits>

namespace cvr {

template <class T> struct VoxTag { typedef T type; };

// kMode: kGroups or kLanes, + kPhong (with Blinn-Phong).
template <typename T, bool TF_LDS, int kMode>
__global__ __launch_bounds__(256) void k_rc1p(RayFrame rf, VolGeom g, const float4* __restrict__ tf, int ntf,
                                               float step, float et, PhongK ph, const float4* __restrict__ grad,
                                               float ka, float kd, QueueShape qs, float4* __restrict__ out,
                                               unsigned long long* __restrict__ counters) {
  __shared__ RayList<kListRays> list;
  extern __shared__ float4 s_tf[];
  if (TF_LDS) {
    stage_tf_padded(s_tf, tf, ntf);
    __syncthreads();
  }
  const float4* tfp = TF_LDS ? s_tf : tf;
  unsigned int nsamp = 0, nshade = 0;
  const f3 eye = ld3(rf.eye);
  auto lit = [&](f3 p) {
    float dd, sp;
    if (!(kMode & kPhong) || !phong_terms(grad, g, ph, p, eye, dd, sp)) return Lit{1.f, 0.f};
    return Lit{ka + kd * dd, ph.ks * sp};
  };
  if constexpr ((kMode & kLanes) != 0) {
    int px, py;
    lane_pixel(rf, qs.first, px, py);
    lane_march<T, TF_LDS, (kMode & kPhong) != 0>(rf, g, tfp, ntf, step, et, px, py, ph.spec, out, nsamp, nshade, lit);
  } else {
    plain_march<T, TF_LDS, (kMode & kPhong) != 0>(rf, g, tfp, ntf, step, et, FramePixels(rf, qs, queue_unit<4>(qs), 4),
                                            ph.spec, list, out, nsamp, nshade, lit);
  }
  if (counters) {
    count_add(counters, 0, nsamp);
    count_add(counters, 1, nshade);
  }
}

int phong_setup(cvr_ctx* c, int on, int gradient_type, float ks, float shininess, const float spec[3],
                const RayFrame& rf, const cvr_light* light, PhongK& ph, hipStream_t st) {
  ph = PhongK{};
  if (!on) return 0;
  if (!(shininess > 0.f)) {
    set_error("cvr_render: Blinn-Phong shininess must be > 0");
    return CVR_ERR_INVALID;
  }
  if (const int rc = build_gradient(c, gradient_type, st)) return rc;
  ph.on = 1;
  ph.ks = ks;
  ph.shininess = shininess;
  for (int i = 0; i < 3; ++i) {
    ph.spec[i] = spec[i];
    // without a light: the camera's own light at the eye (renderingmanager.cpp:421-426)
    ph.lpos[i] = light ? light->position[i] : rf.eye[i];
  }
  return 0;
}

int launch_rc1p(cvr_ctx* c, const RayFrame& rf, const cvr_light* light, float* out, hipStream_t st) {
  const cvr_rc1p_params& P = c->rc1p;
  VolGeom g = geom_of(c);
  float step = P.step_size > 0 ? P.step_size : default_step(c);
  float et = P.et_threshold;
  PhongK ph;
  if (const int rc = phong_setup(c, P.apply_gradient_shading, P.gradient_type, P.ks, P.shininess, P.specular, rf, light,
                                 ph, st))
    return rc;
  const float4* gr = ph.on ? c->d_grad : nullptr;
  bool lds = c->tf_size <= 4096;
  size_t shm = lds ? size_t(c->tf_size + 2) * sizeof(float4) : 0;
  const MarchShape ms = march_shape(rf, g, step, et, ph.on, kLaneRays);
  unsigned long long* cnt = c->collect_stats ? c->d_counters : nullptr;
  float4* o4 = reinterpret_cast<float4*>(out);
  auto launch = [&](auto t, auto l, auto m) {
    using T = typename decltype(t)::type;
    constexpr bool L = decltype(l)::value;
    for_launches(ms.qs, ms.blocks, 256, [&](const QueueShape& qs, int blocks) {
      hipLaunchKernelGGL((k_rc1p<T, L, decltype(m)::value>), dim3(blocks), dim3(256), L ? shm : 0, st, rf, g,
                         c->d_tf_rgbt, c->tf_size, step, et, ph, gr, P.ka, P.kd, qs, o4, cnt);
    });
  };
  auto by_mode = [&](auto t, auto l) {
    with_mode(ms.mode, [&](auto m) { launch(t, l, m); });
  };
  auto by_lds = [&](auto t) {
    if (lds) by_mode(t, std::true_type{});
    else by_mode(t, std::false_type{});
  };
  if (c->dtype == CVR_U8) by_lds(VoxTag<uint8_t>{});
  else by_lds(VoxTag<uint16_t>{});
  CVR_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace cvr
