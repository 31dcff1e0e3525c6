// Directional occlusion shading with cone section tables (gfx950): the renderer of
// RC1PConeTracingDirOcclusionShading.
//
// Host side: the section tables of ConeGaussianSampler::ComputeConeIntegrationSteps
// (rc1pdosct/conegaussiansampler.cpp:212-414) built in FP64: sections are placed along
// the cone axis every d_sigma*sigma (per half interval); the Gaussian sigma doubles
// whenever the cone radius outgrows r_sigma*sigma, and before doubling the cone is
// split into 3 and then 7 narrower sub-cones (circle packings) as the packing limit
// allows.  Each section carries (interval to the next, mip level log2(sigma/sigma0),
// trapezoid half width, amplitude (pr*Ig)^2 / (pi R^2)) with pr the Gaussian's mass
// over the cone diameter by the midpoint rule.
//
// Device side: the march of rc1pdosct/ray_bbox_marching.comp:658-734; each opaque
// sample integrates the occlusion cone towards the eye and (optionally) the shadow
// cone towards the light through the tables (:124-333, :345-562): one Gaussian per
// section on the axis, then 3 then 7 sub-cones that inherit their parent's optical
// depth, trapezoid sums of amplitude * extinction, I = exp(-depth) averaged over the
// sub-cones (the 7-packing weights its ring by the adjacent weight).  The march is
// queue_march's (cvr_queue.hpp; 256^3 at 1024^2 with shadows 41.5 ms a lane per ray, 15.6 queued, 12.6
// with the rows of dos_cone, 10.7 at three wavefronts per SIMD).  A section is the same for all lanes:
// its row and its level's geometry come through scalar loads.
#include "cvr_cone.hpp"
#include "cvr_queue.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace cvr {

// Per-cone constants of the device integration.
struct DosConeK {
  int n1, n3, n7;
  float w, adj7;
  float ax[10][3];  // 3-packing axes, then 7-packing axes, (x, y, z) in the cone frame
};

struct DosK {
  DosConeK occ, sdw;
  const ConeLevel* lev;
  const DosRow* occ_rows;
  const DosRow* sdw_rows;
  int apply_occ, apply_sdw, shadow_type;
  float spot_cos, ka, kd;
  float eye[3], lpos[3], lfwd[3], lup[3], lright[3];
};

// One cone through its section table; sub-cone axes are k*z + uy*y + vx*x.  A section's row is the same
// for all lanes (scalar loads); sections before the first lane leaves the box do without the border
// falloff, which is 1 there.
template <int F, bool kWide>
__device__ __forceinline__ float dos_cone(const void* __restrict__ pyr, const PyrGeom& pg, const DosConeK& C,
                                          const ConeLevel* __restrict__ levels, const DosRow* __restrict__ table,
                                          bool inside, f3 p, f3 k, f3 uy, f3 vx) {
  typedef const __attribute__((address_space(4))) DosRow* ConstRows;
  const ConstRows rows = (ConstRows)(uintptr_t)table;
  const ConstLevels lev = (ConstLevels)(uintptr_t)levels;
  float od[7], lt[7];
  od[0] = 0.f;
  lt[0] = 0.f;
  int i = 0;
  // GetGaussianExtinction (ray_bbox_marching.comp:92-112) of row i at axis d
  auto ext = [&](auto border, int i, f3 d) {
    const f3 tp = p + d * rows[i].track;
    float v = level_read<F, kWide>(pyr, lev + rows[i].level, tp, pg.one);
    if constexpr (decltype(border)::value) v *= border_falloff(pg, tp, rows[i].fall);
    return v * rows[i].amp;
  };
  auto add = [&](int j, int i, float at) {
    od[j] += (lt[j] + at) * rows[i].dint * C.w;
    lt[j] = at;
  };
  // the single-cone sections in groups whose reads are in flight together (256^3 at 1024^2: 15.0 ms
  // with 2, 13.5 with 4, 12.6 with 8, 12.4 with 10, whose remainders cost small volumes more; the
  // 7-packing's registers are more than any of them need)
  constexpr int kAhead = 8;
  const float te = wave_exit(pg, inside, p, k);
  auto group = [&](auto border) {
    float at[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) at[u] = ext(border, i + u, k);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) add(0, i + u, at[u]);
  };
  for (; i + kAhead <= C.n1; i += kAhead) {
    if (rows[i + kAhead - 1].track <= te) group(std::false_type{});
    else group(std::true_type{});
  }
  for (; i < C.n1; ++i) add(0, i, ext(std::true_type{}, i, k));
  if (C.n3 + C.n7 == 0) return __expf(-od[0]);
  od[1] = od[2] = od[0];
  lt[1] = lt[2] = lt[0];
  f3 d3[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) d3[j] = k * C.ax[j][2] + uy * C.ax[j][1] + vx * C.ax[j][0];
  auto sections = [&](auto count, const f3* d, int e) {
    constexpr int kN = decltype(count)::value;
    float t = wave_exit(pg, inside, p, d[0]);
#pragma unroll
    for (int j = 1; j < kN; ++j) t = fminf(t, wave_exit(pg, inside, p, d[j]));
    for (; i < e; ++i) {
      float at[kN];
      if (rows[i].track <= t) {
#pragma unroll
        for (int j = 0; j < kN; ++j) at[j] = ext(std::false_type{}, i, d[j]);
      } else {
#pragma unroll
        for (int j = 0; j < kN; ++j) at[j] = ext(std::true_type{}, i, d[j]);
      }
#pragma unroll
      for (int j = 0; j < kN; ++j) add(j, i, at[j]);
    }
  };
  sections(std::integral_constant<int, 3>{}, d3, i + C.n3);
  if (C.n7 == 0) return (__expf(-od[0]) + __expf(-od[1]) + __expf(-od[2])) / 3.0f;
  // 3 -> 7: each outer cone inherits the depth of the 3-cone it came from, the centre
  // cone their mean (Cone7RayOcclusion, :127-137)
  const float ma = (od[2] + od[1] + od[0]) / 3.0f, mt = (lt[2] + lt[1] + lt[0]) / 3.0f;
  od[6] = od[5] = od[2];
  od[4] = od[3] = od[1];
  od[2] = od[1] = od[0];
  od[0] = ma;
  lt[6] = lt[5] = lt[2];
  lt[4] = lt[3] = lt[1];
  lt[2] = lt[1] = lt[0];
  lt[0] = mt;
  f3 d7[7];
#pragma unroll
  for (int j = 0; j < 7; ++j) d7[j] = k * C.ax[3 + j][2] + uy * C.ax[3 + j][1] + vx * C.ax[3 + j][0];
  sections(std::integral_constant<int, 7>{}, d7, i + C.n7);
  const float ring = __expf(-od[1]) + __expf(-od[2]) + __expf(-od[3]) + __expf(-od[4]) + __expf(-od[5]) + __expf(-od[6]);
  return (__expf(-od[0]) + ring * C.adj7) / (1.0f + C.adj7 * 6.0f);
}

// Shadow cone of ShadowEvaluationKernel (:533-562).  `wp` is the world position.
template <int F, bool kWide>
__device__ __forceinline__ float dos_shadow(const void* __restrict__ pyr, const PyrGeom& pg, const DosK& K, bool inside,
                                            f3 p, f3 wp) {
  f3 k = ld3(K.lfwd), up = ld3(K.lup), right = ld3(K.lright);
  if (K.shadow_type != 2) {
    k = norm3(ld3(K.lpos) - wp);
    if (K.shadow_type == 1 && dot3(k, ld3(K.lfwd)) < K.spot_cos) return 0.f;
    const f3 u1 = norm3(cross3(k, right));
    up = norm3(cross3(k, u1));
    right = u1;
  }
  return dos_cone<F, kWide>(pyr, pg, K.sdw, K.lev, K.sdw_rows, inside, p, k, up, right);
}
// Both terms at p: the occlusion cone along k in the frame (up, right); 0 for one that is off.  The points are
// samples and cells inside the box; kTest asks all the same (k_dos_render).
template <int F, bool kTest = false>
__device__ __forceinline__ void dos_light(const void* __restrict__ pyr, const PyrGeom& pg, const DosK& K, f3 p, f3 wp, f3 k,
                                          f3 up, f3 right, float& Io, float& Is) {
  const bool inside = !kTest || wave_inside(pg, p);
  auto both = [&](auto wide) {
    constexpr bool kWide = decltype(wide)::value;
    Io = K.apply_occ ? dos_cone<F, kWide>(pyr, pg, K.occ, K.lev, K.occ_rows, inside, p, k, up, right) : 0.f;
    Is = K.apply_sdw ? dos_shadow<F, kWide>(pyr, pg, K, inside, p, wp) : 0.f;
  };
  if (pg.wide) both(std::true_type{});
  else both(std::false_type{});
}

// For 8-bit volumes and 32-bit pyramids, rays of their own: with the test of points outside the box the kernel
// takes 162 registers, without it 170, and three wavefronts per SIMD fit up to 168 (256^3 at 1024^2 10.5 and 12.6 ms).
// The others fit without it, and are slower with it (16-bit volume of 168 x 155 x 168 at 760 x 639 2.65 and 2.74 ms).
constexpr int kRays = 4, kShortRays = 16;
template <typename T, int F, int kParts, int kRays>
__global__ __launch_bounds__(256) void k_dos_render(RayFrame rf, VolGeom g, PyrGeom pg, const void* __restrict__ pyr,
                                                    DosK K, const float4* __restrict__ tf, int ntf, float step, float et,
                                                    PhongK ph, const float4* __restrict__ grad, QueueShape qs,
                                                    float4* __restrict__ out,
                                                    unsigned long long* __restrict__ counters) {
  extern __shared__ float4 s_tf[];
  __shared__ WaveQueue<kRays> queue[4];
  if (tile_left_out<kParts>(qs)) return;
  for (int i = threadIdx.x; i < ntf; i += blockDim.x) s_tf[i] = tf[i];
  __syncthreads();
  constexpr bool kTest = sizeof(T) == 1 && F == 0 && kParts == 1;
  const int u = queue_unit<kParts>(qs);
  const f3 eye = ld3(rf.eye);
  const f3 half = mk3(0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]);
  unsigned int nsamp = 0, nshade = 0;
  const float ka = K.apply_occ ? K.ka : 0.f, kd = K.apply_sdw ? K.kd : 0.f;
  const float inv_k = 1.0f / (ka + kd);
  queue_march<T, 64, false, kParts>(rf, g, s_tf, ntf, step, et, qs.rays, FramePixels(rf, qs, u), ph.spec, kParts > 1 ? queue : queue + (threadIdx.x >> 6), out, nsamp, nshade,
                 [&](bool, f3 p, f3 dir) {
                   const f3 wp = p - half;
                   float Io, Is;
                   f3 axis, up, right;
                   occ_frame(dir, axis, up, right);
                   dos_light<F, kTest>(pyr, pg, K, p, wp, norm3(eye - wp), up, right, Io, Is);
                   if (!ph.on) return Lit{inv_k * (Io * ka + Is * kd), 0.f};
                   // Phong branch (:627-643): a sample whose gradient vanishes keeps its colour
                   float dd, sp;
                   if (!phong_terms(grad, g, ph, p, eye, dd, sp)) return Lit{1.f, 0.f};
                   return Lit{inv_k * (Io * ka + Is * kd * dd), Is * (K.apply_sdw ? ph.ks : 0.f) * sp};
                 });
  if (counters) {
    count_add(counters, 0, nsamp);
    count_add(counters, 1, nshade);
  }
}

// Object-space light cache (rc1pdosct/lightcachecomputation.comp:523-546): cell i
// holds (occlusion, shadow) at texture-space position (i + 1/2) * cell, 1 for a term
// that is off.  The occlusion cone turns towards the eye in the frame
// right = normalize(cross(-k, camera up)), up = normalize(cross(k, right)) (:279-291);
// the shadow cone is the renderer's own.  One lane per cell.
template <int F>
__global__ __launch_bounds__(256) void k_lc_dos(PyrGeom pg, const void* __restrict__ pyr, DosK K, f3 cam_up, int rx,
                                                int ry, int rz, f3 cell, f3 half, float2* __restrict__ lc) {
  const size_t n = size_t(rx) * ry * rz;
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int x = int(i % size_t(rx)), y = int((i / size_t(rx)) % size_t(ry)), z = int(i / (size_t(rx) * ry));
  const f3 tp = mk3((float(x) + 0.5f) * cell.x, (float(y) + 0.5f) * cell.y, (float(z) + 0.5f) * cell.z);
  const f3 wp = tp - half;
  const f3 k = norm3(ld3(K.eye) - wp);
  const f3 vr = norm3(cross3(mk3(-k.x, -k.y, -k.z), cam_up));
  float Io, Is;
  dos_light<F>(pyr, pg, K, tp, wp, k, norm3(cross3(k, vr)), vr, Io, Is);
  lc[i] = make_float2(K.apply_occ ? Io : 1.f, K.apply_sdw ? Is : 1.f);
}

// ------------------------------------------------------------------ host: section tables
namespace {
const double kPi = 3.14159265358979323846;
const double kDiv3 = 1.0 + 2.0 / std::sqrt(3.0);  // 3 circles packed in a circle: radius ratio
const double kDiv7 = 3.01;                         // 7 circles (the reference's rounded ratio)

struct Section {
  int ng;
  double pos, radius, sigma;
};

// Mass of N(0, sigma) over [-R, R], midpoint rule on segments of about 0.05.
double gauss_mass(double sigma, double R) {
  const int nt = int(std::ceil((2.0 * R) / 0.05));
  const double seg = (2.0 * R) / double(nt), x0 = -R + 0.5 * seg;
  const double norm = 1.0 / (std::sqrt(2.0 * kPi) * sigma);
  double S = 0.0;
  for (int i = 0; i < nt; ++i) {
    const double x = x0 + seg * double(i);
    S += norm * std::exp(-(x * x) / (2.0 * sigma * sigma)) * seg;
  }
  return S;
}

// Rotation of v by angle t about the unit axis a (Rodrigues), renormalised.
void rotate(const double v[3], double t, const double a[3], double out[3]) {
  const double c = std::cos(t), s = std::sin(t), d = a[0] * v[0] + a[1] * v[1] + a[2] * v[2];
  const double cr[3] = {a[1] * v[2] - a[2] * v[1], a[2] * v[0] - a[0] * v[2], a[0] * v[1] - a[1] * v[0]};
  double r[3], l = 0;
  for (int i = 0; i < 3; ++i) {
    r[i] = v[i] * c + cr[i] * s + a[i] * d * (1.0 - c);
    l += r[i] * r[i];
  }
  l = std::sqrt(l);
  for (int i = 0; i < 3; ++i) out[i] = r[i] / l;
}

struct Builder {
  double half_deg, r_sigma;
  int max_packing, ng = 1;
  std::vector<Section> secs;
  // Places a section at `pos` with sigma `sg`, splitting into more sub-cones (never
  // fewer than the previous section had) while the radius exceeds r_sigma * sg.
  bool add(double pos, double sg) {
    static const double div[3] = {1.0, kDiv3, kDiv7};
    static const int ngs[3] = {1, 3, 7};
    int k = ng == 1 ? 0 : (ng == 3 ? 1 : 2);
    for (;;) {
      ng = ngs[k];
      const double R = pos * std::tan((half_deg / div[k]) * kPi / 180.0);
      if (!(R > r_sigma * sg)) {
        secs.push_back(Section{ng, pos, R, sg});
        return true;
      }
      if (k >= max_packing) return false;
      ++k;
    }
  }
};
}  // namespace

// The clamps of ConeGaussianSampler's setters (conegaussiansampler.cpp:57-172).
static cvr_dos_cone clamp_cone(cvr_dos_cone c, double covered_default) {
  c.half_deg = std::min(std::max(c.half_deg, 0.5f), 89.5f);
  c.max_packing = std::min(std::max(c.max_packing, 0), 2);
  if (!(c.initial_step > 0)) c.initial_step = 0.f;
  const float cov = c.covered_dist > 0 ? c.covered_dist : float(covered_default);
  c.covered_dist = cov > 10.0f ? cov : 10.0f;
  c.d_sigma = std::min(std::max(c.d_sigma, 1.0f), 3.0f);
  c.r_sigma = std::min(std::max(c.r_sigma, 0.5f), 3.0f);
  return c;
}

// The schedule ends only if the Gaussians can outgrow the widest sub-cone allowed: the
// next section sits about d_sigma * sigma further, where that sub-cone's radius grows by
// d_sigma * sigma * tan(half / div); with d_sigma * tan(half / div) >= r_sigma, sigma
// would double without bound.
static bool dos_cone_converges(const cvr_dos_cone& C) {
  static const double div[3] = {1.0, kDiv3, kDiv7};
  const double t = std::tan((double(C.half_deg) / div[C.max_packing]) * kPi / 180.0);
  return double(C.d_sigma) * t < double(C.r_sigma);
}

int dos_build_table(const cvr_dos_cone& C, double sigma0, DosTable& T) {
  if (!(C.initial_step > 0) || !(C.initial_step < C.covered_dist)) {
    set_error("dos params: initial_step must be > 0 and below the covered distance");
    return CVR_ERR_INVALID;
  }
  if (!dos_cone_converges(C)) {
    set_error("dos params: d_sigma * tan(half angle / packing ratio) must stay below r_sigma "
              "(the section schedule would never close)");
    return CVR_ERR_INVALID;
  }
  Builder b{double(C.half_deg), double(C.r_sigma), C.max_packing};
  const double ds = double(C.d_sigma);
  double pos = double(C.initial_step), sg = sigma0;
  std::vector<double> iv;  // interval after each section
  while (!b.add(pos, sg)) sg *= 2.0;
  while (pos < double(C.covered_dist)) {
    double si = ds * sg;
    while (!b.add(pos + si + ds * sg, sg)) sg *= 2.0;
    si += ds * sg;
    iv.push_back(si);
    pos += si;
    if (iv.size() > (1u << 16)) {
      set_error("dos params: more than 65536 cone sections");
      return CVR_ERR_INVALID;
    }
  }
  iv.push_back(0.0);
  const size_t n = b.secs.size();
  T.rows.resize(n);
  T.n[0] = T.n[1] = T.n[2] = 0;
  for (size_t i = 0; i < n; ++i) {
    const Section& s = b.secs[i];
    T.n[s.ng == 1 ? 0 : (s.ng == 3 ? 1 : 2)] += 1;
    const double dint = i == 0 ? s.sigma * std::sqrt(2.0 * kPi) * 0.5 : iv[i - 1] * 0.5;
    const double pr = gauss_mass(s.sigma, s.radius);
    const double Ig = s.sigma * std::sqrt(2.0 * kPi);
    const double amp = (pr * pr) * (Ig * Ig) / (kPi * s.radius * s.radius);
    T.rows[i] = make_float4(float(iv[i]), float(std::log2(s.sigma / sigma0)), float(dint), float(amp));
  }
  // sub-cone axes (conegaussiansampler.cpp:219-252)
  const double z[3] = {0, 0, 1}, y[3] = {0, 1, 0};
  const double half = double(C.half_deg);
  double a[10][3];
  rotate(z, (half - half / kDiv3) * kPi / 180.0, y, a[0]);
  rotate(a[0], 30.0 * kPi / 180.0, z, a[0]);
  rotate(a[0], 120.0 * kPi / 180.0, z, a[1]);
  rotate(a[1], 120.0 * kPi / 180.0, z, a[2]);
  a[3][0] = 0; a[3][1] = 0; a[3][2] = 1;
  rotate(z, (half - half / kDiv7) * kPi / 180.0, y, a[4]);
  for (int j = 5; j < 10; ++j) rotate(a[j - 1], 60.0 * kPi / 180.0, z, a[j]);
  for (int j = 0; j < 10; ++j)
    for (int c = 0; c < 3; ++c) T.axes[j][c] = float(a[j][c]);
  T.adj7 = float(a[4][2]);
  T.init = C.initial_step;
  T.w = C.ui_weight;
  return CVR_OK;
}

static cvr_dos_cone clamp_cone(cvr_dos_cone c, double covered_default);

int check_dos_params(const cvr_dos_params& P) {
  if (!dos_cone_converges(clamp_cone(P.occ, 100.0)) || !dos_cone_converges(clamp_cone(P.sdw, 100.0))) {
    set_error("dos params: d_sigma * tan(half angle / packing ratio) must stay below r_sigma "
              "(the section schedule would never close)");
    return CVR_ERR_INVALID;
  }
  if (P.apply_occlusion == 0 && P.apply_shadow == 0) {
    set_error("dos params: occlusion or shadow must be enabled (the shading divides by ka+kd)");
    return CVR_ERR_INVALID;
  }
  if (!(P.sigma0 > 0) || P.n_levels > kMaxLevels || P.shadow_type < 0 || P.shadow_type > 2 || !(P.et_threshold > 0) ||
      !(P.occ.initial_step > 0) || !(P.sdw.initial_step > 0) || P.density_precision < 0 || P.density_precision > 2) {
    set_error("dos params: sigma0 > 0, n_levels <= 12, shadow_type in {0,1,2}, et_threshold > 0, initial steps > 0, "
              "density_precision 0, 1 or 2");
    return CVR_ERR_INVALID;
  }
  return CVR_OK;
}

int prepare_dos(cvr_ctx* c, const cvr_dos_params& P, hipStream_t st) {
  int rc = check_dos_params(P);
  if (rc) return rc;
  const int bx = P.base_res[0] > 0 ? P.base_res[0] : c->nx;
  const int by = P.base_res[1] > 0 ? P.base_res[1] : c->ny;
  const int bz = P.base_res[2] > 0 ? P.base_res[2] : c->nz;
  rc = build_pyramid(c, bx, by, bz, P.sigma0, P.n_levels, P.density_precision, st);
  if (rc) return rc;
  // SetCoveredDistance(diagonal * 0.50f / 0.75f) in float (dosrcrenderer.cpp:112-113)
  const float diag = volume_diagonal(c);
  const cvr_dos_cone oc = clamp_cone(P.occ, diag * 0.50f), sc = clamp_cone(P.sdw, diag * 0.75f);
  // the tables of the same cones are kept (building and copying them took 0.05 ms of every frame)
  const double sigma0 = P.sigma0;
  const std::vector<ConeLevel> lev = cone_levels(c->pyr);
  if (c->dos_sigma_for == sigma0 && c->dos_lev_for.size() == lev.size() &&
      std::memcmp(c->dos_lev_for.data(), lev.data(), lev.size() * sizeof(ConeLevel)) == 0 && std::memcmp(&c->dos_cones_for[0], &oc, sizeof(oc)) == 0 &&
      std::memcmp(&c->dos_cones_for[1], &sc, sizeof(sc)) == 0)
    return CVR_OK;
  c->dos_sigma_for = 0.0;
  CVR_HIP_CHECK(hipDeviceSynchronize());  // frames in flight may still read the rows
  if ((rc = dos_build_table(oc, P.sigma0, c->dos_occ))) return rc;
  if ((rc = dos_build_table(sc, P.sigma0, c->dos_sdw))) return rc;
  // [levels] [occlusion rows] [shadow rows]
  std::vector<DosRow> rows;
  for (const DosTable* T : {&c->dos_occ, &c->dos_sdw}) {
    float track = T->init;
    for (const float4& r : T->rows) {
      const double level = double(r.y);  // log2(sigma / sigma0), a whole number
      DosRow d{track, r.z, r.w, float(-0.5 * 1.4426950408889634 * std::exp2(-2.0 * level)), 0, {0, 0, 0}};
      d.level = std::min(std::max(int(std::lround(level)), 0), c->pyr.levels - 1);
      rows.push_back(d);
      track += r.x;
    }
  }
  const size_t lb = lev.size() * sizeof(ConeLevel), rb = rows.size() * sizeof(DosRow);
  if ((rc = sized_buffer(&c->d_dos_rows, &c->dos_rows_bytes, lb + rb))) {
    if (rc == CVR_ERR_NOMEM) set_error("dos: out of device memory");
    return rc;
  }
  std::vector<char> buf(lb + rb);
  std::memcpy(buf.data(), lev.data(), lb);
  std::memcpy(buf.data() + lb, rows.data(), rb);
  CVR_HIP_CHECK(hipMemcpy(c->d_dos_rows, buf.data(), buf.size(), hipMemcpyHostToDevice));
  c->dos_lev_for = lev;
  c->dos_cones_for[0] = oc;
  c->dos_cones_for[1] = sc;
  c->dos_sigma_for = sigma0;
  return CVR_OK;
}

static DosConeK cone_k(const DosTable& T) {
  DosConeK k{};
  k.n1 = T.n[0];
  k.n3 = T.n[1];
  k.n7 = T.n[2];
  k.w = T.w;
  k.adj7 = T.adj7;
  std::memcpy(k.ax, T.axes, sizeof(k.ax));
  return k;
}

int launch_dos(cvr_ctx* c, const RayFrame& rf, const cvr_light* light, float* out, hipStream_t st) {
  const cvr_dos_params& P = c->dos;
  int rc = prepare_dos(c, P, st);
  if (rc) return rc;
  DosK K{};
  K.occ = cone_k(c->dos_occ);
  K.sdw = cone_k(c->dos_sdw);
  K.lev = static_cast<const ConeLevel*>(c->d_dos_rows);
  K.occ_rows = reinterpret_cast<const DosRow*>(K.lev + kMaxLevels);
  K.sdw_rows = K.occ_rows + c->dos_occ.rows.size();
  K.apply_occ = P.apply_occlusion;
  K.apply_sdw = P.apply_shadow;
  K.shadow_type = P.shadow_type;
  K.spot_cos = float(std::cos(double(P.spot_max_deg) * kPi / 180.0));
  K.ka = P.ka;
  K.kd = P.kd;
  for (int i = 0; i < 3; ++i) {
    K.eye[i] = rf.eye[i];
    // without a light: the camera's own light (renderingmanager.cpp:421-426)
    K.lpos[i] = light ? light->position[i] : rf.eye[i];
    K.lfwd[i] = light ? light->forward[i] : -rf.f[i];
    K.lup[i] = light ? light->up[i] : rf.u[i];
    K.lright[i] = light ? light->right[i] : rf.s[i];
  }
  VolGeom g = geom_of(c);
  const float step = P.step_size > 0 ? P.step_size : default_step(c);
  const size_t shm = size_t(c->tf_size) * sizeof(float4);
  if (shm > 64 * 1024) { set_error("dos renderer: transfer function larger than 4096 entries"); return CVR_ERR_UNSUPPORTED; }
  PhongK ph;
  if ((rc = phong_setup(c, P.apply_phong, P.gradient_type, P.ks, P.shininess, P.specular, rf, light, ph, st))) return rc;
  if (P.light_cache) {
    // PreComputeLightCache (dosrcrenderer.cpp:555-651), then the object-space march
    if ((rc = lc_prepare(c, P.light_cache_res))) return rc;
    const int rx = c->lc_res[0], ry = c->lc_res[1], rz = c->lc_res[2];
    const int dims[3] = {c->nx, c->ny, c->nz}, res[3] = {rx, ry, rz};
    const float sc[3] = {c->sx, c->sy, c->sz};
    float cs[3];
    for (int i = 0; i < 3; ++i) cs[i] = sc[i] * (float(dims[i]) / float(res[i]));  // VolumeScales * (dims / res)
    const size_t n = size_t(rx) * ry * rz;
    const f3 cam_up{rf.u[0], rf.u[1], rf.u[2]};
    const f3 half{0.5f * g.G[0], 0.5f * g.G[1], 0.5f * g.G[2]};
    const f3 cell{cs[0], cs[1], cs[2]};
    with_fmt(c->pyr.fmt, [&](auto f) {
      hipLaunchKernelGGL((k_lc_dos<decltype(f)::value>), dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, c->pyr,
                         c->d_pyr_oct, K, cam_up, rx, ry, rz, cell, half, c->d_lc);
    });
    CVR_HIP_CHECK(hipGetLastError());
    return launch_lc_render(c, rf, P.apply_occlusion, P.apply_shadow, P.ka, P.kd, step, P.et_threshold, ph, out, st);
  }
  unsigned long long* cnt = c->collect_stats ? c->d_counters : nullptr;
  float4* o4 = reinterpret_cast<float4*>(out);
  // small frames: workgroups whose wavefronts share their rays (256^3 at 100^2 0.24 ms, 0.45 with rays of
  // their own; 200 x 150 0.43 and 0.76; 256^2 0.92 and 1.07, 128^3 0.40 either way; 400 x 300 1.28 and 1.38;
  // 512^2 3.30 and 3.02; 1024^2 12.7 and 10.7)
  const bool shared = size_t(rf.W) * rf.H < (1 << 16);
  QueueShape shape = queue_shape(rf.W, rf.H, kRays, shared ? 4 : 1, shared ? 64 : 256);
  if ((rc = short_tiles(c, rf, step, P.et_threshold, 1024, st, &shape.short_tiles))) return rc;
  with_types(c->dtype, c->pyr.fmt, [&](auto t, auto f) {
    using T = typename decltype(t)::type;
    auto launch = [&](const QueueShape& s, auto parts, auto rays) {
      for_launches(s, s.blocks, 256, [&](const QueueShape& qs, int blocks) {
        hipLaunchKernelGGL((k_dos_render<T, decltype(f)::value, decltype(parts)::value, decltype(rays)::value>), dim3(blocks),
                           dim3(256), shm, st, rf, g, c->pyr, c->d_pyr_oct, K, c->d_tf_rgbt, c->tf_size, step,
                           P.et_threshold, ph, c->d_grad, qs, o4, cnt);
      });
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, kRays> few;
    if (shared) launch(shape, std::integral_constant<int, 4>{}, few);
    else launch(shape, one, few);
    if (shape.short_tiles) launch(short_shape(rf, shape, kShortRays), one, std::integral_constant<int, kShortRays>{});
  });
  CVR_HIP_CHECK(hipGetLastError());
  return CVR_OK;
}

}  // namespace cvr
