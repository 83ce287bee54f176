// Visibility, sun occlusion and single-ray queries on a scene.
#include "wide.h"

namespace flux {

template <typename Query, bool kShare>
__global__ void __launch_bounds__(256, 5) k_query(flux_scene S, Query q, int64_t total,
                                                  int64_t block) {
  __shared__ int stack[4][kStackRows][64];
  IndexSource<Query> src;
  src.init(q, total, block);
  trace_wave<kShare>(S, src, &stack[threadIdx.x >> 6][0][threadIdx.x & 63]);
}

// Queries of up to this many rays share the walks that are left once a wave
// has handed out its rays: such a query lasts as long as its longest walk
// and leaves the VALUs idle.  One sun over 10,368 facets: 69 us without
// sharing, 32 with; over 41,472: 105 and 47.  With 25 rays a wave (124,416)
// 135 and 94; with 50 (248,832) sharing costs instructions that the chip has
// no time for (150 and 190).
constexpr int64_t kShareRays = 131072;

template <typename Query>
static int launch_query(const flux_scene *scene, const Query &q, int64_t total, hipStream_t st) {
  const int64_t block = trace_block(total);
  const dim3 grid(trace_groups((total + block - 1) / block));
  if (total <= kShareRays)
    hipLaunchKernelGGL((k_query<Query, true>), grid, dim3(256), 0, st, *scene, q, total, block);
  else
    hipLaunchKernelGGL((k_query<Query, false>), grid, dim3(256), 0, st, *scene, q, total, block);
  FLUX_LAUNCH_CHECK();
  return 0;
}

// Facet-to-facet visibility of the pairs (p, q), row by row: consecutive
// rays share their source facet.
template <typename T>
struct VisQuery {
  const int64_t *I, *J;
  int64_t n;
  int mode;
  const T *P;
  uint8_t *out;

  __device__ __forceinline__ void begin(const flux_scene &S, LaneRay &L, int64_t r) const {
    const int64_t p = r / n, i64 = I[p], j64 = J[r - p * n];
    L.cur = kLaneBlocked;
    if (i64 < 0 || i64 >= S.nf || j64 < 0 || j64 >= S.nf) return;
    const int i = (int)i64, j = (int)j64;
    T pi[3] = {0, 0, 0}, pj[3] = {0, 0, 0};
    if (mode == FLUX_MODE_EMBREE)
      for (int c = 0; c < 3; ++c) {
        pi[c] = P[i64 * 3 + c];
        pj[c] = P[j64 * 3 + c];
      }
    pair_begin(S, L, i, j, mode, pi, pj);
  }
  __device__ __forceinline__ void end(const flux_scene &, int64_t r, bool blocked) const {
    out[r] = blocked ? 0 : 1;
  }
};

// The ray from facet f towards a direction d: CGAL mode from the FP64
// centroid, facet skipped (aabb_wrapper.cpp:95-108); EMBREE mode from
// P + 1e-3 N, nothing skipped (shape.py:400-421).
template <typename T>
__device__ __forceinline__ void sun_begin(const flux_scene &S, LaneRay &L, int64_t f,
                                          const double *dir, int mode, const T *P, const T *N) {
  double o[3], d[3] = {dir[0], dir[1], dir[2]};
  int skip = -1;
  if (mode == FLUX_MODE_CGAL) {
    for (int c = 0; c < 3; ++c) o[c] = S.cen[f * 3 + c];
    skip = (int)f;
  } else {
    embree_sun_ray(P + f * 3, N + f * 3, dir, o, d);
  }
  ray_setup(L.r, o, d);
  // the walk ends where the ray leaves the scene along its main axis
  const double lo = sel3(S.box, L.r.kz), hi = sel3(S.box + 3, L.r.kz);
  const double tmax = fmax(((L.r.Sz < 0.0 ? lo : hi) - L.r.o[2]) * L.r.Sz, 0.0);
  lane_begin(S, L, o, d, tmax, INFINITY, 0x7fffffff, skip, -1);
  // Along an infinite component every triangle is at t = 0, which has no
  // place in a range of t / tmax: such a ray takes the stackless walk alone.
  if (L.r.Sz == 0.0) {
    L.cur = kLaneVisible;
    L.flags |= kFlagLost;
  }
}

// Occlusion of facet I[p] towards D[q] (or D[p]): all facets of one
// direction after the other, so a wave's rays run in parallel.
template <typename T>
struct OccQuery {
  const int64_t *I;
  int64_t m;
  const double *D;
  int64_t M;
  int per_face, mode;
  const T *Nrm, *P;
  uint8_t *out;

  __device__ __forceinline__ void begin(const flux_scene &S, LaneRay &L, int64_t r) const {
    const int64_t q = r / m, p = r - q * m, f = I[p];
    L.cur = kLaneVisible;
    if (f < 0 || f >= S.nf) return;
    sun_begin(S, L, f, D + (per_face ? p : q) * 3, mode, P, Nrm);
  }
  __device__ __forceinline__ void end(const flux_scene &, int64_t r, bool blocked) const {
    const int64_t q = r / m, p = r - q * m;
    out[per_face ? p : p * M + q] = blocked ? 1 : 0;
  }
};

// E[f, k] = F0 * max(0, N_f . d_k) if facet f sees sun k, else 0: the 1-D
// sun branch of get_direct_irradiance (shape.py:224-226) for M suns at once.
// The dot product is taken in FP64 (N . Dsun of a mesh-dtype N with an FP64
// direction promotes to FP64 in NumPy) and stored in the mesh dtype.  The
// rays go out sun by sun in Morton order of the facets: neighbours in a wave
// walk the same nodes.
template <typename T>
struct IrradianceQuery {
  const T *Nrm, *P;
  const double *D;  // NULL: the one direction `sun`
  int64_t M;
  double F0;
  int mode;
  T *E;
  double sun[3];

  __device__ __forceinline__ void direction(int64_t k, double d[3]) const {
    for (int c = 0; c < 3; ++c) d[c] = D ? D[k * 3 + c] : sun[c];
  }

  __device__ __forceinline__ void begin(const flux_scene &S, LaneRay &L, int64_t r) const {
    const int64_t k = r / S.nf;
    double d[3];
    direction(k, d);
    sun_begin(S, L, S.order[r - k * S.nf], d, mode, P, Nrm);
  }
  __device__ __forceinline__ void end(const flux_scene &S, int64_t r, bool blocked) const {
    const int64_t k = r / S.nf, f = S.order[r - k * S.nf];
    double d[3], nf3[3];
    direction(k, d);
    load3(Nrm, f, nf3);
    const double cosi = (nf3[0] * d[0] + nf3[1] * d[1]) + nf3[2] * d[2];
    E[f * M + k] = blocked ? (T)0 : (T)(F0 * (cosi > 0.0 ? cosi : 0.0));
  }
};

__global__ void k_intersect1(flux_scene S, const double *__restrict__ x,
                             const double *__restrict__ d, int64_t nr,
                             int64_t *__restrict__ hit, double *__restrict__ xt) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nr) return;
  double o[3] = {x[k * 3], x[k * 3 + 1], x[k * 3 + 2]};
  double dd[3] = {d[k * 3], d[k * 3 + 1], d[k * 3 + 2]};
  Ray64 r;
  ray_setup(r, o, dd);
  RayBox rb;
  raybox_setup(rb, o, dd);
  double t;
  int h = closest_hit(S, r, rb, -1, &t);
  hit[k] = h;
  for (int c = 0; c < 3; ++c) xt[k * 3 + c] = h >= 0 ? o[c] + t * dd[c] : 0.0;
}

}  // namespace flux

using namespace flux;

static int direct_irradiance(const flux_scene *scene, const void *P, const void *Nrm, int dtype,
                             const double *D, const double *sun, int64_t M, double F0, int mode,
                             void *E, void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_direct_irradiance: NULL scene");
  FLUX_CHECK(M >= 0, "flux_direct_irradiance: negative M");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_direct_irradiance: bad dtype");
  FLUX_CHECK(mode == FLUX_MODE_CGAL || mode == FLUX_MODE_EMBREE,
             "flux_direct_irradiance: bad mode");
  const int64_t total = scene->nf * M;
  if (total == 0) return 0;
  FLUX_CHECK(Nrm && (D || sun) && E && (mode == FLUX_MODE_CGAL || P),
             "flux_direct_irradiance: NULL array");
  hipStream_t st = as_stream(stream);
  const double s[3] = {sun ? sun[0] : 0.0, sun ? sun[1] : 0.0, sun ? sun[2] : 0.0};
  if (dtype == FLUX_F64)
    return launch_query(scene,
                        IrradianceQuery<double>{(const double *)Nrm, (const double *)P, D, M, F0,
                                                mode, (double *)E, {s[0], s[1], s[2]}},
                        total, st);
  return launch_query(scene,
                      IrradianceQuery<float>{(const float *)Nrm, (const float *)P, D, M, F0, mode,
                                             (float *)E, {s[0], s[1], s[2]}},
                      total, st);
}

extern "C" int flux_direct_irradiance(const flux_scene *scene, const void *P, const void *Nrm,
                                      int dtype, const double *D, int64_t M, double F0,
                                      int mode, void *E, void *stream) {
  return direct_irradiance(scene, P, Nrm, dtype, D, nullptr, M, F0, mode, E, stream);
}

// The direction travels with the launch: the copy of 24 bytes that a time
// step started with held the host for 15 us and the GPU idle for about 35.
extern "C" int flux_direct_irradiance_sun(const flux_scene *scene, const void *P, const void *Nrm,
                                          int dtype, const double *sun, double F0, int mode,
                                          void *E, void *stream) {
  return direct_irradiance(scene, P, Nrm, dtype, nullptr, sun, 1, F0, mode, E, stream);
}

extern "C" int flux_vis_mn(const flux_scene *scene, const int64_t *I, int64_t m,
                           const int64_t *J, int64_t n, int mode, const void *P,
                           int dtype, uint8_t *out, void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_vis_mn: NULL scene");
  FLUX_CHECK(m >= 0 && n >= 0, "flux_vis_mn: negative sizes");
  FLUX_CHECK(mode == FLUX_MODE_CGAL || mode == FLUX_MODE_EMBREE, "flux_vis_mn: bad mode %d",
             mode);
  FLUX_CHECK(mode == FLUX_MODE_CGAL || P != nullptr, "flux_vis_mn: EMBREE mode needs P");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_vis_mn: bad dtype");
  if (m == 0 || n == 0) return 0;
  FLUX_CHECK(I && J && out, "flux_vis_mn: NULL array");
  FLUX_CHECK(m <= (int64_t)65535 * 65535, "flux_vis_mn: m too large");
  hipStream_t st = as_stream(stream);
  if (dtype == FLUX_F64)
    return launch_query(scene, VisQuery<double>{I, J, n, mode, (const double *)P, out}, m * n,
                        st);
  return launch_query(scene, VisQuery<float>{I, J, n, mode, (const float *)P, out}, m * n, st);
}

extern "C" int flux_occluded(const flux_scene *scene, const int64_t *I, int64_t m,
                             const double *D, int64_t M, int per_face, int mode,
                             const void *P, const void *Nrm, int dtype, uint8_t *out,
                             void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_occluded: NULL scene");
  FLUX_CHECK(m >= 0 && M >= 0, "flux_occluded: negative sizes");
  FLUX_CHECK(mode == FLUX_MODE_CGAL || mode == FLUX_MODE_EMBREE,
             "flux_occluded: bad mode %d", mode);
  FLUX_CHECK(!per_face || M == m, "flux_occluded: per_face needs M == m");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_occluded: bad dtype");
  if (m == 0 || M == 0) return 0;
  FLUX_CHECK(I && D && out, "flux_occluded: NULL array");
  FLUX_CHECK(mode == FLUX_MODE_CGAL || (Nrm != nullptr && P != nullptr),
             "flux_occluded: EMBREE mode needs P and N");
  hipStream_t st = as_stream(stream);
  const int64_t total = m * (per_face ? 1 : M);
  if (dtype == FLUX_F64)
    return launch_query(scene,
                        OccQuery<double>{I, m, D, M, per_face, mode, (const double *)Nrm,
                                         (const double *)P, out},
                        total, st);
  return launch_query(scene,
                      OccQuery<float>{I, m, D, M, per_face, mode, (const float *)Nrm,
                                      (const float *)P, out},
                      total, st);
}

extern "C" int flux_intersect1(const flux_scene *scene, const double *x, const double *d,
                               int64_t n_rays, int64_t *hit_index, double *xt,
                               void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_intersect1: NULL scene");
  FLUX_CHECK(n_rays >= 0, "flux_intersect1: negative size");
  if (n_rays == 0) return 0;
  FLUX_CHECK(x && d && hit_index && xt, "flux_intersect1: NULL array");
  const int TB = 256;
  hipLaunchKernelGGL(k_intersect1, dim3(ceil_div_u(n_rays, TB)), dim3(TB), 0,
                     as_stream(stream), *scene, x, d, n_rays, hit_index, xt);
  FLUX_LAUNCH_CHECK();
  return 0;
}
