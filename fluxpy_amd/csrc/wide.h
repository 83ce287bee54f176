// Four-wide BVH and the wave-scheduled any-hit traversal behind the
// form-factor mask, the visibility matrix and the sun queries.
//
// A walk of the binary preorder layouts (ray.h) takes about 80 dependent
// node loads per facet-to-facet ray of a terrain, and in a wave of such
// walks nearly every step has a few lanes at a leaf, so the FP64 triangle
// test runs with 3 or 4 of 64 lanes active.  Here
//  * a node holds the quantised boxes of up to four children in 64 bytes
//    (one cache line segment, four 16-byte loads), which cuts the dependent
//    loads per ray to about 21 nodes + 5 triangles;
//  * each lane is at a node, at a leaf or without work, and every iteration
//    of the wave runs one of the two steps, for the larger group;
//  * lanes whose ray has ended take new rays once a quarter of the wave is
//    out of work, instead of waiting for the longest ray of 64;
//  * in small queries, which last as long as their longest walk, lanes
//    without work take deferred children off other lanes' stacks.
//
// Decisions do not depend on any of this: the set of triangles tested always
// contains every triangle the FP64 test hits on the queried segment (the
// quantised boxes contain the padded FP32 boxes), and a query's answer is a
// property of that set.
#pragma once
#include "ray.h"

namespace flux {

// Child codes: >= 0 a wide node, < 0 the leaf of triangle ~code.  Lane
// states below every leaf code (facet counts are below 2^30):
constexpr int kLaneIdle = INT32_MIN;         // no ray
constexpr int kLaneVisible = INT32_MIN + 1;  // walk ended without a blocker
constexpr int kLaneBlocked = INT32_MIN + 2;  // a blocker was found
constexpr int kLaneDone = INT32_MIN + 2;     // states <= kLaneDone have no step to run

// Deferred children per lane (LDS, 256 B per entry and wave) and the room
// for a node's writes past them.  Terrains of 41k facets reach 14, a walk
// that would need more marks itself and is repeated on the stackless layout.
constexpr int kWideStack = 24;
constexpr int kStackRows = kWideStack + 3;
// Out-of-work lanes that trigger a refill: a refill's ray set-up costs about
// one node step, whatever the number of lanes it serves.
constexpr int kRefill = 16;

// Steps between two rounds of sharing, and the lanes without work that one
// needs (trace_share).  A round costs about as much as a third of a step:
// one sun over 10,368 facets takes 32 us with a round after every step, 37
// after two, 55 after four; 33 with 8 lanes and 36 with 32.
constexpr int kShareSteps = 1;
constexpr int kShareIdle = 16;
static_assert(kShareSteps >= 1, "the walk goes on between two rounds");

// kFlagHelper: the lane walks a part of the ray of lane flags >> 8.
enum : int { kFlagPair = 1, kFlagReverse = 2, kFlagLost = 4, kFlagHelper = 8 };

struct LaneRay {
  Ray64 r;
  // slab tests run in t / tmax, so that the walked part of the ray is 0 .. 1:
  // plane p is at p inv - oi
  float inv[3], oi[3];
  int oct;       // 3 x the direction octant
  double tlim;   // hits at (t, k) before (tlim, klim) block
  int klim;
  int skip1, skip2;
  int cur, flags;
  int sp;        // deferred children, in LDS words
};

// Walk the ray up to tmax (finite).  The direction is scaled in FP64, where
// its length does not matter.  Rounding of a plane's position, in units of
// 2^-24 of the scene's scale: the FP32 origin 1, the reciprocal direction
// over tmax 4, inv x origin 1, the two fused steps 2.  The node
// boxes contain boxes padded by 16 units, so a triangle hit at t in 0 .. tlim
// has a slab interval of positive length inside 0 .. 1.
__device__ __forceinline__ void lane_begin(const flux_scene &S, LaneRay &L, const double o[3],
                                           const double d[3], double tmax, double tlim, int klim,
                                           int skip1, int skip2) {
  const double scale = tmax * (1.0 + 1e-5);
  int oct = 0;
  for (int c = 0; c < 3; ++c) {
    const float dc = (float)(d[c] * scale);
    const bool neg = dc < 0.0f;
    const float iv = fminf(fabsf(1.0f / dc), S.inv_max);
    L.inv[c] = neg ? -iv : iv;
    L.oi[c] = (float)o[c] * L.inv[c];
    oct += neg ? 3 << c : 0;
  }
  L.oct = oct;
  L.tlim = tlim;
  L.klim = klim;
  L.skip1 = skip1;
  L.skip2 = skip2;
  L.sp = 0;
  L.cur = S.root;
}

// The ray that decides whether facet i sees facet j; a pair decided without
// a walk leaves the lane visible or blocked.
//   CGAL mode (aabb_wrapper.cpp:64-93): origin = FP64 centroid of i,
//   direction = centroid_j - centroid_i, i skipped, visible iff j is the
//   closest hit; i == j -> false.
//   EMBREE mode (shape.py:349-398): the ray of embree_pair_ray from the
//   model centroids Pi, Pj (read in this mode only), nothing skipped,
//   visible iff j is the closest hit.
template <typename T>
__device__ __forceinline__ void pair_begin(const flux_scene &S, LaneRay &L, int i, int j,
                                           int mode, const T *Pi, const T *Pj) {
  double o[3], d[3];
  int skip = -1;
  L.cur = kLaneBlocked;
  if (mode == FLUX_MODE_CGAL) {
    if (i == j) return;
    const double *ci = S.cen + (int64_t)i * 3, *cj = S.cen + (int64_t)j * 3;
    for (int c = 0; c < 3; ++c) {
      o[c] = ci[c];
      d[c] = cj[c] - ci[c];
    }
    skip = i;
  } else if (!embree_pair_ray(Pi, Pj, o, d)) {
    L.cur = kLaneVisible;
    return;
  }
  ray_setup(L.r, o, d);
  const double tj = tri_hit(L.r, S.tri + (int64_t)j * 9);
  if (tj >= 0.0) lane_begin(S, L, o, d, tj, tj, j, skip, j);
}

__device__ __forceinline__ void lane_pop(LaneRay &L, const int *stk) {
  if (L.sp > 0) {
    L.sp -= 64;
    L.cur = stk[L.sp];
  } else {
    L.cur = kLaneVisible;
  }
}

// t / tmax of a quantised plane (byte c of w), clamped to the walked part.
__device__ __forceinline__ float plane(uint32_t w, int c, float s, float b) {
  return __builtin_amdgcn_fmed3f(fmaf((float)((w >> (8 * c)) & 0xffu), s, b), 0.0f, 1.0f);
}

// The lane's node: test the four children, go on with the first one in the
// node's order for the ray's octant and defer the others that are hit (stk:
// the lane's column of the wave's stack).  About 110 VALU instructions:
// every deferral is an unconditional LDS write below a pointer that moves
// only past hits, so the order needs no loop over slots and no branches.
__device__ __forceinline__ void lane_node(const flux_scene &S, LaneRay &L, int *stk) {
  const uint4 *nd = S.wide + (int64_t)L.cur * 4;
  const uint4 n0 = nd[0], n1 = nd[1], n2 = nd[2], n3 = nd[3];
  const int ex = (int)n0.w;
  const float sx = __builtin_amdgcn_ldexpf(L.inv[0], (int)(int8_t)ex);
  const float sy = __builtin_amdgcn_ldexpf(L.inv[1], (int)(int8_t)(ex >> 8));
  const float sz = __builtin_amdgcn_ldexpf(L.inv[2], (int)(int8_t)(ex >> 16));
  const float bx = fmaf(__uint_as_float(n0.x), L.inv[0], -L.oi[0]);
  const float by = fmaf(__uint_as_float(n0.y), L.inv[1], -L.oi[1]);
  const float bz = fmaf(__uint_as_float(n0.z), L.inv[2], -L.oi[2]);
  const bool gx = L.inv[0] < 0.0f, gy = L.inv[1] < 0.0f, gz = L.inv[2] < 0.0f;
  const uint32_t ax = gx ? n2.w : n2.x, fx = gx ? n2.x : n2.w;
  const uint32_t ay = gy ? n3.x : n2.y, fy = gy ? n2.y : n3.x;
  const uint32_t az = gz ? n3.y : n2.z, fz = gz ? n2.z : n3.y;
  int c[4] = {(int)n1.x, (int)n1.y, (int)n1.z, (int)n1.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float tn =
        fmaxf(fmaxf(plane(ax, k, sx, bx), plane(ay, k, sy, by)), plane(az, k, sz, bz));
    const float tf =
        fminf(fminf(plane(fx, k, sx, bx), plane(fy, k, sy, by)), plane(fz, k, sz, bz));
    c[k] = tn < tf ? c[k] : kLaneIdle;
  }
  const uint32_t ord = n3.z >> L.oct;
  const bool w0 = ord & 2u, w1 = ord & 4u, wp = ord & 1u;
  const int a0 = w0 ? c[1] : c[0], a1 = w0 ? c[0] : c[1];
  const int b0 = w1 ? c[3] : c[2], b1 = w1 ? c[2] : c[3];
  const int d0 = wp ? b0 : a0, d1 = wp ? b1 : a1, d2 = wp ? a0 : b0, d3 = wp ? a1 : b1;
  int sp = L.sp;
  stk[sp] = d3;
  sp += d3 != kLaneIdle ? 64 : 0;
  stk[sp] = d2;
  sp += d2 != kLaneIdle ? 64 : 0;
  stk[sp] = d1;
  sp += d1 != kLaneIdle ? 64 : 0;
  if (sp > kWideStack * 64) {
    sp = kWideStack * 64;
    L.flags |= kFlagLost;
  }
  L.sp = sp;
  L.cur = d0;
  if (d0 == kLaneIdle) lane_pop(L, stk);
}

// The lane's leaf, for queries that stop at the first blocker.
__device__ __forceinline__ void lane_leaf(const flux_scene &S, LaneRay &L, const int *stk) {
  const int t = ~L.cur;
  bool block = false;
  if (t != L.skip1 && t != L.skip2) {
    const double th = tri_hit(L.r, S.tri + (int64_t)t * 9);
    block = th >= 0.0 && (th < L.tlim || (th == L.tlim && t < L.klim));
  }
  if (block)
    L.cur = kLaneBlocked;
  else
    lane_pop(L, stk);
}

// What a triangle says about a line that is walked in one direction (origin
// centroid i, end centroid j) and could be walked from j to i instead.
// Both directions compute the same edge functions but for rounding: the
// origin and the sheared coordinates differ by at most 16 u L (u = 2^-53, L
// the scene's extent; |S| <= 1), so each of U, V, W differs by less than
// 152 u L^2, and edge_tol = 2^-42 L^2 is more than twelve times that.  With
// t' = 1 - t, t differs by at most edge_tol (|Az| + |Bz| + |Cz| + 4) / |det|.
//  kMiss    the line passes outside, both ways
//  kThrough it passes inside at t, known to 2^-12 both ways
//  kUnsure  rounding may decide
enum : int { kMiss = 0, kThrough = 1, kUnsure = 2 };

__device__ __forceinline__ int tri_sides(const Ray64 &r, const TriEdges &e, double tol,
                                         double *t) {
  const double hi = fmax(fmax(e.U, e.V), e.W), lo = fmin(fmin(e.U, e.V), e.W);
  if (hi > tol && lo < -tol) return kMiss;
  if (!(lo > tol || hi < -tol)) return kUnsure;
  const double det = e.U + e.V + e.W;
  const double Az = r.Sz * e.A_z, Bz = r.Sz * e.B_z, Cz = r.Sz * e.C_z;
  *t = (e.U * Az + e.V * Bz + e.W * Cz) / det;
  return tol * (fabs(Az) + fabs(Bz) + fabs(Cz) + 4.0) <= 0x1p-12 * fabs(det) ? kThrough : kUnsure;
}

constexpr double kEndBand = 0x1p-10;  // t this close to 0 or 1 decides nothing

// The ray i -> j for both directions at once (kFlagPair), if both facets
// are hit clearly at the ends; else for i -> j alone, with j -> i to follow
// (kFlagReverse).
__device__ __forceinline__ void both_begin(const flux_scene &S, LaneRay &L, int i, int j,
                                           bool both) {
  double o[3], d[3];
  const double *ci = S.cen + (int64_t)i * 3, *cj = S.cen + (int64_t)j * 3;
  for (int c = 0; c < 3; ++c) {
    o[c] = ci[c];
    d[c] = cj[c] - ci[c];
  }
  ray_setup(L.r, o, d);
  const double tj = tri_hit(L.r, S.tri + (int64_t)j * 9);
  L.flags = 0;
  if (both) {
    double ti = 2.0, te = 2.0;
    const bool ok =
        tri_sides(L.r, tri_edges(L.r, S.tri + (int64_t)i * 9), S.edge_tol, &ti) == kThrough &&
        tri_sides(L.r, tri_edges(L.r, S.tri + (int64_t)j * 9), S.edge_tol, &te) == kThrough &&
        fabs(ti) < 0.5 * kEndBand && fabs(te - 1.0) < 0.5 * kEndBand;
    L.flags = ok ? kFlagPair : kFlagReverse;
  }
  L.skip1 = i;
  L.skip2 = j;
  L.cur = kLaneBlocked;
  if (tj >= 0.0) lane_begin(S, L, o, d, tj, tj, j, i, j);
}

// The lane's leaf in such a walk.  A blocker that is clear of the ends and
// of its own edges blocks both directions; any other triangle that is not a
// clear miss leaves the reverse direction to a walk of its own.
__device__ __forceinline__ void both_leaf(const flux_scene &S, LaneRay &L, const int *stk) {
  const int t = ~L.cur;
  bool block = false;
  if (t != L.skip1 && t != L.skip2) {
    const TriEdges e = tri_edges(L.r, S.tri + (int64_t)t * 9);
    const double U = e.U, V = e.V, W = e.W;
    const bool mixed = (U < 0.0 || V < 0.0 || W < 0.0) && (U > 0.0 || V > 0.0 || W > 0.0);
    const double det = U + V + W;
    const double Az = L.r.Sz * e.A_z, Bz = L.r.Sz * e.B_z, Cz = L.r.Sz * e.C_z;
    const double th = (U * Az + V * Bz + W * Cz) / det;
    block = !mixed && det != 0.0 && th >= 0.0 && (th < L.tlim || (th == L.tlim && t < L.klim));
    if (L.flags & kFlagPair) {
      const double hi = fmax(fmax(U, V), W), lo = fmin(fmin(U, V), W);
      const bool miss = hi > S.edge_tol && lo < -S.edge_tol;
      const bool thru = (lo > S.edge_tol || hi < -S.edge_tol) &&
                        S.edge_tol * (fabs(Az) + fabs(Bz) + fabs(Cz) + 4.0) <=
                            0x1p-12 * fabs(det);
      const bool inside = thru && th > kEndBand && th < 1.0 - kEndBand;
      const bool beyond = thru && (th < -kEndBand || th > 1.0 + kEndBand);
      if (inside)
        L.flags &= ~kFlagReverse;
      else if (!miss && !beyond)
        L.flags |= kFlagReverse;
    }
  }
  if (block)
    L.cur = kLaneBlocked;
  else
    lane_pop(L, stk);
}

// A walk that ran out of stack has skipped children: once it has ended,
// repeat it on the stackless layout unless it found a blocker anyway.  Rays
// are handed out while other lanes walk: those keep their mark, and the
// lanes that take new rays have none.
__device__ __forceinline__ void lane_recover(const flux_scene &S, LaneRay &L) {
  if (L.cur == kLaneVisible && (L.flags & kFlagLost)) {
    // the ray's box test again, from the shears
    double o[3] = {0.0, 0.0, 0.0}, d[3] = {0.0, 0.0, 0.0};
    const double dz = 1.0 / L.r.Sz;
    for (int c = 0; c < 3; ++c) {
      if (c == L.r.kx) o[c] = L.r.o[0], d[c] = L.r.Sx * dz;
      if (c == L.r.ky) o[c] = L.r.o[1], d[c] = L.r.Sy * dz;
      if (c == L.r.kz) o[c] = L.r.o[2], d[c] = dz;
    }
    RayBox rb;
    raybox_setup(rb, o, d);
    if (any_blocker(S, L.r, rb, L.tlim, L.klim, L.skip1, L.skip2)) L.cur = kLaneBlocked;
    if (L.flags & kFlagPair) L.flags |= kFlagReverse;
  }
  if (L.cur <= kLaneDone) L.flags &= ~kFlagLost;
}

// LDS written by some lanes of the wave is read by others (the wave's LDS
// operations complete in order; this keeps the compiler's order too).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Index of this lane among the set lanes of m.
__device__ __forceinline__ int lane_rank(uint64_t m) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Helpers that are done, and lanes at a ray that is known to be blocked,
// hand in what they found: the lane that owns the ray (the one that refill
// gave it to) takes it over, the helpers are free again.  What several lanes
// found of a pair's ray adds up like what one lane finds: a blocker of both
// directions decides both, else any of them may ask for the reverse walk.
__device__ __forceinline__ void share_report(LaneRay &L, int *stk) {
  enum : int { kBlocked = 1, kReverse = 2, kBothBlocked = 4 };
  const int lane = threadIdx.x & 63;
  int *found = stk - lane + kWideStack * 64;  // rows past the deferred children
  const bool helper = L.flags & kFlagHelper;
  const bool done = L.cur <= kLaneDone && L.cur != kLaneIdle && !(L.flags & kFlagLost);
  int bits = 0;
  if (done && L.cur == kLaneBlocked)
    bits = (L.flags & (kFlagPair | kFlagReverse)) == kFlagPair ? kBlocked | kBothBlocked
                                                               : kBlocked;
  if (done && (L.flags & kFlagReverse)) bits |= kReverse;
  found[lane] = helper ? 0 : bits;
  wave_lds_order();
  const int own = helper ? L.flags >> 8 : lane;
  if (helper && bits) atomicOr(&found[own], bits);
  wave_lds_order();
  const int all = found[own];
  if (helper) {
    if (done || (all & kBlocked)) {
      L.cur = kLaneIdle;
      L.flags = 0;
    }
  } else if (L.cur != kLaneIdle) {
    if (all & kBlocked) L.cur = kLaneBlocked;
    if (L.flags & kFlagPair) {
      if (all & kBothBlocked)
        L.flags &= ~kFlagReverse;
      else if (all & kReverse)
        L.flags |= kFlagReverse;
    }
  }
  wave_lds_order();
}

template <typename V>
__device__ __forceinline__ void take_from(V &v, int lane) {
  v = __shfl(v, lane);
}

// Lanes without work take the first deferred child (the largest part left)
// of lanes that have one, with their rays.
__device__ __forceinline__ void trace_share(LaneRay &L, int *stk) {
  share_report(L, stk);
  const int lane = threadIdx.x & 63;
  int *donor = stk - lane + kWideStack * 64, *child = donor + 64;
  const uint64_t idle = __ballot(L.cur == kLaneIdle);
  const bool can = L.cur > kLaneDone && L.sp > 0;
  const uint64_t give = __ballot(can);
  const int count = min(__popcll(idle), __popcll(give));
  if (count == 0) return;
  if (can) {
    const int k = lane_rank(give);
    if (k < count) {
      donor[k] = lane;
      child[k] = stk[0];
      L.sp -= 64;
      stk[0] = stk[L.sp];
    }
  }
  wave_lds_order();
  const int k = lane_rank(idle);
  const bool take = L.cur == kLaneIdle && k < count;
  const int from = take ? donor[k] : lane;
  const int cur = take ? child[k] : L.cur, sp = take ? 0 : L.sp;
  const int flags = take ? 0 : L.flags;
  for (int c = 0; c < 3; ++c) {
    take_from(L.r.o[c], from);
    take_from(L.inv[c], from);
    take_from(L.oi[c], from);
  }
  take_from(L.r.Sx, from);
  take_from(L.r.Sy, from);
  take_from(L.r.Sz, from);
  take_from(L.r.kx, from);
  take_from(L.r.ky, from);
  take_from(L.r.kz, from);
  take_from(L.oct, from);
  take_from(L.tlim, from);
  take_from(L.klim, from);
  take_from(L.skip1, from);
  take_from(L.skip2, from);
  const int f = __shfl(L.flags, from);
  L.flags = take ? (f & (kFlagPair | kFlagReverse)) | kFlagHelper |
                       (f & kFlagHelper ? f & ~0xff : from << 8)
                 : flags;
  L.cur = cur;
  L.sp = sp;
  wave_lds_order();
}

// The wave's loop.  src.refill(S, L) ends the rays of done lanes, hands new
// ones out and returns false once no lane of the wave has one and none are
// left; src.drained() says that none are left to hand out (from then on
// refill runs only when every lane is done, and so has every helper).
template <bool kShare, typename Src>
__device__ __forceinline__ void trace_wave(const flux_scene &S, Src &src, int *stk) {
  LaneRay L;
  L.cur = kLaneIdle;
  L.sp = 0;
  L.flags = 0;
  int steps = 0;
  while (true) {
    const int nn = __popcll(__ballot(L.cur >= 0));
    const int nl = __popcll(__ballot(L.cur < 0 && L.cur > kLaneDone));
    if (nn + nl == 0 || (nn + nl <= 64 - kRefill && !src.drained())) {
      lane_recover(S, L);
      if (kShare && __ballot(L.flags & kFlagHelper)) share_report(L, stk);
      if (!src.refill(S, L)) break;
      continue;
    }
    // no rays left: the ones under way are walked by all lanes (the last
    // refill of a wave follows when the last lane is done)
    if (kShare && nn + nl <= 64 - kShareIdle && --steps < 0) {
      steps = kShareSteps;
      trace_share(L, stk);
      continue;
    }
    if (nn >= nl) {
      if (L.cur >= 0) lane_node(S, L, stk);
    } else {
      if (L.cur < 0 && L.cur > kLaneDone) src.leaf(S, L, stk);
    }
  }
}

// Rays numbered 0 .. total - 1 for trace_wave: a wave takes blocks of
// `block` consecutive rays, `nwaves` blocks apart.  Query::begin sets up ray
// r and Query::end stores its answer (every ray has begin, then end).
template <typename Query>
struct IndexSource {
  Query q;
  int64_t total, block, stride, base, next, stop;
  int64_t ray;  // the lane's

  __device__ __forceinline__ void init(const Query &query, int64_t n, int64_t blk) {
    q = query;
    total = n;
    block = blk;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    stride = (((int64_t)gridDim.x * blockDim.x) >> 6) * blk;
    base = wave * blk;
    next = min(base, total);
    stop = min(base + blk, total);
    ray = 0;
  }

  __device__ __forceinline__ bool drained() const { return next >= stop; }

  __device__ __forceinline__ bool refill(const flux_scene &S, LaneRay &L) {
    if (L.cur == kLaneVisible || L.cur == kLaneBlocked) q.end(S, ray, L.cur == kLaneBlocked);
    if (L.cur <= kLaneDone) L.cur = kLaneIdle;
    const uint64_t idle = __ballot(L.cur == kLaneIdle);
    const int want = __popcll(idle);
    const int rank = L.cur == kLaneIdle ? lane_rank(idle) : -1;
    int given = 0;
    while (given < want && next < stop) {
      const int take = (int)min((int64_t)(want - given), stop - next);
      if (rank >= given && rank < given + take) {
        ray = next + (rank - given);
        q.begin(S, L, ray);
      }
      given += take;
      next += take;
      if (next >= stop) {
        base += stride;
        next = min(base, total);
        stop = min(base + block, total);
      }
    }
    return given > 0 || __ballot(L.cur > kLaneIdle) != 0;
  }

  __device__ __forceinline__ void leaf(const flux_scene &S, LaneRay &L, const int *stk) {
    lane_leaf(S, L, stk);
  }
};

// Rays per block: a full wave's, or fewer so that a small query spreads over
// the chip (its time is its longest walk, which lanes at other steps delay).
static inline int64_t trace_block(int64_t total) {
  const int64_t b = total / (1280 * 4);
  return b < 8 ? 8 : (b < 64 ? b : 64);
}

// Workgroups of four waves that fill the chip (20 waves a CU: 102 VGPRs and
// 8 KB of LDS each), or as many as there is work for.
static inline unsigned trace_groups(int64_t wave_items) {
  const int64_t g = (wave_items + 3) / 4;
  return (unsigned)(g < 1 ? 1 : (g < 1280 ? g : 1280));
}

}  // namespace flux
