// srf_trace_dev.h -- device helpers shared by the traversal kernels
// (srf_trace.hip) and the two-level scene kernels (srf_scene.hip).
#pragma once

#include <float.h>
#include <math.h>

#include "srf_internal.h"

namespace srf {
namespace {

constexpr int kTraceBlock = 128;
constexpr int kTraceStack = kMaxBranchLevels;  // see above
constexpr uint32_t kDone = 0xffffffffu;

struct RaySetup {
  float o[3], d[3], inv[3];
  int sign[3];
  uint32_t sbits;  // sign[k] << k, so the near child needs no indexed load
};

__device__ __forceinline__ RaySetup setup_ray(const srf_ray *rays, uint32_t i, uint32_t &flags,
                                              uint32_t &prev) {
  const float4 *r4 = reinterpret_cast<const float4 *>(rays + i);
  float4 a = r4[0], b = r4[1];
  RaySetup s;
  s.o[0] = a.x;
  s.o[1] = a.y;
  s.o[2] = a.z;
  s.d[0] = b.x;
  s.d[1] = b.y;
  s.d[2] = b.z;
  flags = __float_as_uint(a.w);
  prev = __float_as_uint(b.w);
  for (int k = 0; k < 3; k++) {
    s.sign[k] = s.d[k] < 0.0f ? 1 : 0;
    // (float)(1.0 / dir): correctly rounded float division gives the same bits
    s.inv[k] = 1.0f / s.d[k];
  }
  s.sbits = (uint32_t)s.sign[0] | ((uint32_t)s.sign[1] << 1) | ((uint32_t)s.sign[2] << 2);
  return s;
}

// IntersectRayAABB, render/render_accel_triangle.cc:1815-1861 (two-box
// nodes, tmax clamped to maxT) and render/render_accel_tetra.cc:1934-1978
// (own box, tmin <= maxT).
template <bool kClampTmax>
__device__ __forceinline__ bool ray_aabb(const RaySetup &s, float maxT, float bx0, float by0,
                                         float bz0, float bx1, float by1, float bz1) {
  float mnx = s.sign[0] ? bx1 : bx0, mxx = s.sign[0] ? bx0 : bx1;
  float mny = s.sign[1] ? by1 : by0, mxy = s.sign[1] ? by0 : by1;
  float mnz = s.sign[2] ? bz1 : bz0, mxz = s.sign[2] ? bz0 : bz1;
  float tminx = (mnx - s.o[0]) * s.inv[0];
  float tmaxx = (mxx - s.o[0]) * s.inv[0];
  float tminy = (mny - s.o[1]) * s.inv[1];
  float tmaxy = (mxy - s.o[1]) * s.inv[1];
  float tmin = (tminx > tminy) ? tminx : tminy;
  float tmax = (tmaxx < tmaxy) ? tmaxx : tmaxy;
  float tminz = (mnz - s.o[2]) * s.inv[2];
  float tmaxz = (mxz - s.o[2]) * s.inv[2];
  tmin = (tmin > tminz) ? tmin : tminz;
  tmax = (tmax < tmaxz) ? tmax : tmaxz;
  if (kClampTmax) {
    tmax = (maxT < tmax) ? maxT : tmax;
    return (tmax > 0.0f) && (tmin <= tmax);
  }
  return (tmax > 0.0f) && (tmin <= tmax) && (tmin <= maxT);
}

// The same test for a wavefront whose rays all have the direction signs
// `sb` (sign[k] << k, wavefront-uniform) and a node loaded through the
// scalar unit: the near and far planes are chosen once for the wavefront
// (scalar selects) instead of per lane; the arithmetic is ray_aabb's.
template <bool kClampTmax>
__device__ __forceinline__ bool ray_aabb_wave(const RaySetup &s, uint32_t sb, float maxT,
                                              float bx0, float by0, float bz0, float bx1,
                                              float by1, float bz1) {
  const float mnx = (sb & 1u) ? bx1 : bx0, mxx = (sb & 1u) ? bx0 : bx1;
  const float mny = (sb & 2u) ? by1 : by0, mxy = (sb & 2u) ? by0 : by1;
  const float mnz = (sb & 4u) ? bz1 : bz0, mxz = (sb & 4u) ? bz0 : bz1;
  float tminx = (mnx - s.o[0]) * s.inv[0];
  float tmaxx = (mxx - s.o[0]) * s.inv[0];
  float tminy = (mny - s.o[1]) * s.inv[1];
  float tmaxy = (mxy - s.o[1]) * s.inv[1];
  float tmin = (tminx > tminy) ? tminx : tminy;
  float tmax = (tmaxx < tmaxy) ? tmaxx : tmaxy;
  float tminz = (mnz - s.o[2]) * s.inv[2];
  float tmaxz = (mxz - s.o[2]) * s.inv[2];
  tmin = (tmin > tminz) ? tmin : tminz;
  tmax = (tmax < tmaxz) ? tmax : tmaxz;
  if (kClampTmax) {
    tmax = (maxT < tmax) ? maxT : tmax;
    return (tmax > 0.0f) && (tmin <= tmax);
  }
  return (tmax > 0.0f) && (tmin <= tmax) && (tmin <= maxT);
}

// The box test where no NaN can arise: the ray's origin and the reciprocals
// finite and not zero (plain_ray), every box finite (BuildParams::odd_box is
// zero). Choosing the later of two entries by a comparison, as the reference
// does, or by the hardware's maximum then gives the same values, and three
// go in one instruction: 17 in place of 28 for a box with its planes chosen
// (nx.. the nearer, fx.. the farther ones). The exit must lie above zero, so
// the smallest float above zero joins the entries. Heightfield 512, 1024^2
// rays 595 -> 555 us; 1M lines 4.93 -> 4.82 ms; solids 1 %. The sphere kernels
// keep the comparisons: nothing gained for occlusion rays, and the closest-hit
// kernel spills more registers (9.0 -> 9.2 ms).
__device__ __forceinline__ bool plain_ray(const RaySetup &s) {
  bool ok = true;
  for (int k = 0; k < 3; k++)
    ok = ok && fabsf(s.o[k]) <= FLT_MAX && fabsf(s.inv[k]) <= FLT_MAX && s.inv[k] != 0.0f;
  return ok;
}
__device__ __forceinline__ bool box_plain(const RaySetup &s, float maxT, float nx, float ny,
                                          float nz, float fx, float fy, float fz) {
  const float a = (nx - s.o[0]) * s.inv[0], b = (ny - s.o[1]) * s.inv[1],
              c = (nz - s.o[2]) * s.inv[2];
  const float d = (fx - s.o[0]) * s.inv[0], e = (fy - s.o[1]) * s.inv[1],
              f = (fz - s.o[2]) * s.inv[2];
  const float enter = fmaxf(fmaxf(fmaxf(a, b), c), __uint_as_float(1u));
  return enter <= fminf(fminf(fminf(d, e), f), maxT);
}
// Both boxes of a node for lanes of the signs sb (wavefront-uniform), searched
// up to maxT.
__device__ __forceinline__ void boxes_plain(const RaySetup &s, uint32_t sb, float maxT,
                                            const float4 &n0, const float4 &n1, const float4 &n2,
                                            bool &h0, bool &h1) {
  const bool x = sb & 1u, y = sb & 2u, z = sb & 4u;
  h0 = box_plain(s, maxT, x ? n1.z : n0.x, y ? n1.w : n0.y, z ? n2.x : n0.z, x ? n0.x : n1.z,
                 y ? n0.y : n1.w, z ? n0.z : n2.x);
  h1 = box_plain(s, maxT, x ? n2.y : n0.w, y ? n2.z : n1.x, z ? n2.w : n1.y, x ? n0.w : n2.y,
                 y ? n1.x : n2.z, z ? n1.y : n2.w);
}

// ---------------------------------------------------- rays of a wavefront
//
// A wavefront carries 2^lg rays: 64 where a launch has enough of them to fill
// the chip, fewer below that (wave_rays). Fewer rays share a shorter walk, so
// a small launch, which is as long as its longest wavefronts, ends sooner; its
// idle lanes cost nothing and take part in paired and queued tests. Rays that
// will mostly be traced one by one, a lane each, want their wavefronts full
// at smaller launches: where fewer than half of the 2^lg parts of a run of
// 2^lg_alone rays share direction signs, the run stays in one wavefront, and
// those of its other parts leave (250k random rays on 8k triangles: 158 us in
// wavefronts of 64, 310 us in 16s). The grid holds the first parts of all runs,
// then the second ones and so on: blocks that leave are together at its end
// (with a run's parts in neighbouring blocks the ones that stay fall on every
// fourth CU: 450 us).
struct WaveRays {
  uint32_t lg, lg_alone;  // lg <= lg_alone
  uint32_t singles;       // whether lanes that share with none are worth a walk each
};
// blocks that one part of every run takes
__host__ __device__ __forceinline__ uint32_t wave_run_blocks(uint64_t n, WaveRays w) {
  const uint32_t lg = w.lg_alone + 31 - __builtin_clz(kTraceBlock / 64);
  return (uint32_t)((n + (1ull << lg) - 1) >> lg);
}
struct WaveRay {
  uint32_t i;  // this lane's ray
  bool first;  // the lane stands for its ray (the others repeat one)
  bool own;    // and writes its result
};
// False for a wavefront without rays. The lanes beyond the wavefront's rays,
// and the last one's beyond n, repeat a ray: the paired and queued leaf tests
// want all 64 lanes.
template <uint32_t kRuns = 4>
__device__ __forceinline__ bool wave_ray(const srf_ray *__restrict__ rays, uint32_t n, WaveRays w,
                                         WaveRay &r) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t lg = w.lg;
  uint32_t block = xcd_block<kRuns>(), part_no = 0;
  const uint32_t lg_parts = w.lg_alone - lg;
  const uint32_t run_blocks = wave_run_blocks(n, w);
  for (; part_no < (1u << lg_parts) && block >= run_blocks; part_no++) block -= run_blocks;
  if (part_no >> lg_parts) return false;
  const uint64_t from = (uint64_t)__builtin_amdgcn_readfirstlane(
                            block * (kTraceBlock / 64) + (threadIdx.x >> 6))
                        << w.lg_alone;
  const uint64_t base = from + ((uint64_t)part_no << lg);
  if (base >= n) return false;
  if (lg_parts) {
    const uint32_t run = 1u << w.lg_alone, part = 1u << lg;
    const uint64_t k = from + (lane & (run - 1u));
    const float *d = rays[k < n ? k : n - 1].dir;
    const uint64_t x = __ballot(d[0] < 0.0f), y = __ballot(d[1] < 0.0f), z = __ballot(d[2] < 0.0f);
    uint32_t same = 0;
    for (uint32_t at = 0; at < run; at += part) {
      const uint64_t m = (part == 64u ? ~0ull : (1ull << part) - 1ull) << at;
      same += ((x & m) == 0 || (x & m) == m) && ((y & m) == 0 || (y & m) == m) &&
              ((z & m) == 0 || (z & m) == m);
    }
    if (2 * same < run / part) {
      if (base != from) return false;
      lg = w.lg_alone;
    }
  }
  const uint32_t count = 1u << lg;
  const uint32_t j = (uint32_t)base + (lane & (count - 1u));
  r.i = j < n ? j : n - 1;
  r.first = lane < count;
  r.own = r.first && j < n;
  return true;
}

// A launch of wavefront walks leaves the rays it has no group for to a second
// launch by a mark in their hits (no hit has a negative t), so that the two
// can spread their rays over wavefronts each as it wants.
constexpr float kAlone = -1.0f;
__device__ __forceinline__ void leave_alone(srf_hit *__restrict__ hits, const WaveRay &r) {
  if (r.own) hits[r.i].t = kAlone;
}
// The second launch's ray, 2^lg of a wavefront: false for a lane without one.
__device__ __forceinline__ bool ray_alone(const srf_hit *__restrict__ hits, uint32_t n,
                                          uint32_t lg, WaveRay &r) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = xcd_block() * (kTraceBlock / 64) + (threadIdx.x >> 6);
  const uint64_t i = ((uint64_t)wave << lg) + lane;
  r.i = (uint32_t)i;
  r.first = r.own = true;
  return (lane >> lg) == 0 && i < n && hits[i].t == kAlone;
}

// ------------------------------------------------------- wavefront groups
//
// A wavefront traversal (one walk for many lanes, nodes and primitives loaded
// through the scalar unit) needs its lanes to share direction signs. A
// wavefront of mixed signs -- the tiles a camera's axes cross, and the ones
// that a frame of odd width lets run over a row's end -- is walked once per
// group of lanes that share signs and stay close together; only lanes in no
// such group are traced one by one. Tracing them all one by one left a few
// wavefronts running alone at the end of a launch (a lane's dependent vector
// loads take about 1 us each): 2048^2 rays on 16M spheres spent 6.2 of 21.0 ms
// there (17.1 -> 13.4 ms a call by groups), 512 x 384 rays on 2M spheres 1.9
// of 3.6 ms (6.2 -> 4.0 ms with the rebuild); solids and lines 0-2 %.
constexpr int kGroupTries = 8;  // groups of one wavefront that are looked for
constexpr int kGroupMin = 8;    // lanes of a group worth a walk of its own when
                                // more groups than that are needed

// Origins of a group lie within this of each other.
__device__ __forceinline__ float group_reach(const BuildParams *__restrict__ P) {
  float e = 0.0f;
  for (int k = 0; k < 3; k++) e = fmaxf(e, P->root_bmax[k] - P->root_bmin[k]);
  return 0.02f * e;
}

// The lanes of `todo` that share the signs of its first lane and lie close
// to it: origins within `reach`, directions within a quarter (14 degrees) of
// the largest component.
__device__ __forceinline__ uint64_t next_group(const RaySetup &s, uint64_t todo, float reach) {
  const int lead = __builtin_ctzll(todo);
  auto of = [&](float x) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lead));
  };
  bool same = s.sbits == (uint32_t)__builtin_amdgcn_readlane((int)s.sbits, lead);
  const float d0 = of(s.d[0]), d1 = of(s.d[1]), d2 = of(s.d[2]);
  const float tol = 0.25f * fmaxf(fabsf(d0), fmaxf(fabsf(d1), fabsf(d2)));
  same = same && fabsf(s.d[0] - d0) <= tol && fabsf(s.d[1] - d1) <= tol &&
         fabsf(s.d[2] - d2) <= tol;
  same = same && fabsf(s.o[0] - of(s.o[0])) <= reach && fabsf(s.o[1] - of(s.o[1])) <= reach &&
         fabsf(s.o[2] - of(s.o[2])) <= reach;
  return (__ballot(same) & todo) | (1ull << lead);
}

// The number of this lane's group, -1 for a lane that is traced alone, -2 for
// one that repeats another's ray (`first` false). Lanes of one sign are group
// 0. Up to kGroupTries groups are kept whatever their sizes; where the lanes
// do not fit in so many, only groups of kGroupMin lanes or more, and where they
// need more than half of them, no single lanes without `singles`.
__device__ __forceinline__ int wave_group(const RaySetup &s, float reach, bool first,
                                          bool singles) {
  const uint32_t sb = __builtin_amdgcn_readfirstlane(s.sbits);
  if (__all(s.sbits == sb)) return first ? 0 : -2;
  uint64_t todo = __ballot(first);
  const int lane = threadIdx.x & 63;
  int group = -1, size = 0, groups = 0;
  for (int g = 0; g < kGroupTries && todo; g++) {
    const uint64_t m = next_group(s, todo, reach);
    todo &= ~m;
    groups++;
    if ((m >> lane) & 1u) {
      group = g;
      size = __popcll(m);
    }
  }
  if (!first) return -2;
  const int least = todo ? kGroupMin : (groups > kGroupTries / 2 && !singles ? 2 : 1);
  return size < least ? -1 : group;
}

// Calls walk(mask) (uniform control flow) for each group of a wavefront.
template <class Walk>
__device__ __forceinline__ void walk_groups(int group, Walk walk) {
  for (int g = 0; g < kGroupTries; g++) {
    const uint64_t m = __ballot(group == g);
    if (m) walk(m);
  }
}

// Orders a wavefront's own LDS writes before its reads (LDS operations of one
// wavefront run in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Leaf tests put off and run 64 at a time. A walk whose visits do not depend
// on the hits found (solids and lines are never narrowed) appends a (lane,
// primitive) entry for each test and runs them in rounds of 64, one entry a
// lane, so that all lanes test whatever the number of lanes that reach a leaf.
// A round's entries are in each ray's own visiting order. key[] keeps each
// ray's best so far as (t bits, rank) with the smallest winning; rank is
// kQueueSettled for earlier rounds' hits, so a rank below it wins ties with
// them and one above loses.
constexpr uint32_t kQueueLeaf = 4;  // primitives of one append
constexpr uint32_t kQueueSettled = 0x80000000u;
struct LeafQueue {  // one wavefront's part of the block's LDS
  float4 org[64];   // origin, previous primitive
  float4 dir[64];
  unsigned long long key[64];
  uint32_t best[64];  // primitive of key
  uint32_t prim[64 * kQueueLeaf + 64];
  uint8_t lane[64 * kQueueLeaf + 64];
};
__device__ __forceinline__ unsigned long long queue_key(float t, uint32_t rank) {
  return ((unsigned long long)__float_as_uint(t + 0.0f) << 32) | rank;  // -0 orders as 0
}
__device__ __forceinline__ void queue_start(LeafQueue &Q, const RaySetup &s, uint32_t prev) {
  const int l = threadIdx.x & 63;
  Q.org[l] = make_float4(s.o[0], s.o[1], s.o[2], __uint_as_float(prev));
  Q.dir[l] = make_float4(s.d[0], s.d[1], s.d[2], 0.0f);
  Q.key[l] = queue_key(FLT_MAX, kQueueSettled);
  Q.best[l] = SRF_NO_PRIM;
}
// Runs one entry a lane: entry l of prim / lane where l < cnt. test(s, prim,
// prev, rank, t): whether the ray s hits, at which t, and its rank, given the
// entry's number in the round.
template <class Test>
__device__ __forceinline__ void queue_round(LeafQueue &Q, const uint32_t *prim,
                                            const uint8_t *lane, uint32_t cnt, Test test) {
  const uint32_t l = threadIdx.x & 63u;
  bool hit = false;
  uint32_t r = 0, q = 0;
  unsigned long long key = 0;
  if (l < cnt) {
    q = prim[l];
    r = lane[l];
    const float4 a = Q.org[r], b = Q.dir[r];
    RaySetup s;
    s.o[0] = a.x;
    s.o[1] = a.y;
    s.o[2] = a.z;
    s.d[0] = b.x;
    s.d[1] = b.y;
    s.d[2] = b.z;
    uint32_t rank = l;
    float t = 0.0f;
    hit = test(s, q, __float_as_uint(a.w), rank, t);
    key = queue_key(t, rank);
  }
  if (__ballot(hit)) {
    if (hit) atomicMin(&Q.key[r], key);
    wave_lds_sync();
    if (hit && Q.key[r] == key) Q.best[r] = q;
    wave_lds_sync();
    Q.key[l] = (Q.key[l] & ~0xffffffffull) | kQueueSettled;
    wave_lds_sync();
  }
}
// Moves entries [at, cnt) (fewer than 64 of them) to the front.
__device__ __forceinline__ uint32_t queue_keep(uint32_t *prim, uint8_t *lane, uint32_t at,
                                               uint32_t cnt) {
  const uint32_t l = threadIdx.x & 63u, rest = cnt > at ? cnt - at : 0u;
  if (at && rest) {
    uint32_t q = 0, r = 0;
    if (l < rest) {
      q = prim[at + l];
      r = lane[at + l];
    }
    wave_lds_sync();
    if (l < rest) {
      prim[l] = q;
      lane[l] = (uint8_t)r;
    }
  }
  return rest;
}
// Runs the entries in rounds of 64 (`all`: the last, partial one too) and
// keeps the rest.
template <class Test>
__device__ __forceinline__ void queue_run(LeafQueue &Q, uint32_t &cnt, bool all, Test test) {
  uint32_t at = 0;
  wave_lds_sync();
  while (cnt >= at + 64u || (all && cnt > at)) {
    queue_round(Q, Q.prim + at, Q.lane + at, cnt - at, test);
    at += 64u;
  }
  cnt = queue_keep(Q.prim, Q.lane, at, cnt);
}

// Appends primitives [q0, q1) for the lanes of `mask`; run() is called when
// 64 entries or more wait.
template <class Run>
__device__ __forceinline__ void queue_leaf(LeafQueue &Q, uint32_t &cnt, uint64_t mask, uint32_t q0,
                                           uint32_t q1, Run run) {
  const uint32_t l = threadIdx.x & 63u;
  const bool in = (mask >> l) & 1u;
  const uint32_t rank = __popcll(mask & ((1ull << l) - 1ull)), lanes = __popcll(mask);
  for (uint32_t q = q0; q < q1; q += kQueueLeaf) {
    const uint32_t c = min(q1 - q, kQueueLeaf);
    if (in)
      for (uint32_t k = 0; k < c; k++) {
        Q.prim[cnt + rank * c + k] = q + k;
        Q.lane[cnt + rank * c + k] = (uint8_t)l;
      }
    cnt += lanes * c;
    if (cnt >= 64u) run();
  }
}

// ---------------------------------------------------------------- triangles

// TriangleIsect (Moller-Trumbore), render/render_accel_triangle.cc:1887-1938,
// on a packed triangle (p0, e1 = p1 - p0, e2 = p2 - p0). u, v and t are the
// reference's expressions; the estimates ue/ve/te (numerator x hardware
// reciprocal, within ~4e-7 relative of the exact values) only reject
// triangles the exact comparisons would reject as well. kEPS >= 1e-30 keeps
// det normal, so the reciprocal estimate is accurate.
__device__ __forceinline__ bool tri_isect(const RaySetup &s, float4 A, float4 B, float4 C,
                                          bool double_sided, float kEPS, bool filter,
                                          float tin, float &tout, float &uout, float &vout) {
  const float e1x = B.x, e1y = B.y, e1z = B.z, e2x = C.x, e2y = C.y, e2z = C.z;
  const float dx = s.d[0], dy = s.d[1], dz = s.d[2];
  float px = dy * e2z - dz * e2y;
  float py = dz * e2x - dx * e2z;
  float pz = dx * e2y - dy * e2x;
  float det = (e1x * px + e1y * py) + e1z * pz;
  if (double_sided) {
    if (fabsf(det) < kEPS) return false;
  } else {
    if (det < kEPS) return false;
  }
  float sx = s.o[0] - A.x, sy = s.o[1] - A.y, sz = s.o[2] - A.z;
  float un = (sx * px + sy * py) + sz * pz;
  const float rc = __builtin_amdgcn_rcpf(det);
  const float ue = un * rc;
  if (filter && (ue < -1e-5f || ue > 1.00001f)) return false;
  float qx = sy * e1z - sz * e1y;
  float qy = sz * e1x - sx * e1z;
  float qz = sx * e1y - sy * e1x;
  float vn = (qx * dx + qy * dy) + qz * dz;
  const float ve = vn * rc;
  if (filter && (ve < -1e-5f || ue + ve > 1.00001f)) return false;
  float tn = (e2x * qx + e2y * qy) + e2z * qz;
  const float te = tn * rc;
  if (filter && (te < -1e-30f || te > tin * 1.00001f)) return false;
  float inv_det = 1.0f / det;  // correctly rounded: equals (float)(1.0 / det)
  float u = un * inv_det;
  float v = vn * inv_det;
  float t = tn * inv_det;
  if (u < 0.0f || u > 1.0f) return false;
  if (v < 0.0f || u + v > 1.0f) return false;
  if (t < 0.0f || t > tin) return false;
  tout = t;
  uout = u;
  vout = v;
  return true;
}

// Empty asm that takes the three values as operands: their loads are issued
// here, together, instead of being sunk past the branch that follows (one
// memory round trip instead of two).
__device__ __forceinline__ void keep_loaded(const float4 &a, const float4 &b, const float4 &c) {
  asm volatile("" ::"v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z),
               "v"(b.w), "v"(c.x), "v"(c.y), "v"(c.z), "v"(c.w));
}

// The same for values loaded through the scalar unit (wavefront-uniform
// addresses): the loads are issued together and waited for once, and the
// values stay in scalar registers.
__device__ __forceinline__ void keep_loaded_s(const float4 &a, const float4 &b, const float4 &c) {
  asm volatile("" ::"s"(a.x), "s"(a.y), "s"(a.z), "s"(a.w), "s"(b.x), "s"(b.y), "s"(b.z),
               "s"(b.w), "s"(c.x), "s"(c.y), "s"(c.z), "s"(c.w));
}

__device__ __forceinline__ void keep_loaded_s2(const float4 &a, const float4 &b) {
  asm volatile("" ::"s"(a.x), "s"(a.y), "s"(a.z), "s"(a.w), "s"(b.x), "s"(b.y), "s"(b.z),
               "s"(b.w));
}

// A lane's pending far children in LDS, kStride entries apart (one column
// per lane, so a wavefront's accesses never share a bank row twice).
template <int kStride>
struct Stack32 {
  uint32_t *w;
  __device__ __forceinline__ void put(int k, uint32_t x) const { w[k * kStride] = x; }
  __device__ __forceinline__ uint32_t get(int k) const { return w[k * kStride]; }
};
// The same for node indices below 2^24: the low 16 and the high 8 bits in two
// planes, 3 bytes per entry instead of 4, so that 8 wavefronts per SIMD fit in
// the LDS (measured on the heightfield: 1.57 -> 1.48 ms).
template <int kStride>
struct Stack24 {
  uint16_t *lo;
  uint8_t *hi;
  __device__ __forceinline__ void put(int k, uint32_t x) const {
    lo[k * kStride] = (uint16_t)x;
    hi[k * kStride] = (uint8_t)(x >> 16);
  }
  __device__ __forceinline__ uint32_t get(int k) const {
    return (uint32_t)lo[k * kStride] | ((uint32_t)hi[k * kStride] << 16);
  }
};

// Closest hit (kAny: any hit closer than tlimit) of one ray against a
// triangle accelerator, TriangleAccel::Traverse
// (render/render_accel_triangle.cc:2511-2669). `st` is this lane's stack
// (Stack32 or Stack24). Returns whether an occluder was found (kAny);
// t/u/v/prim receive the closest hit (t = FLT_MAX, prim = SRF_NO_PRIM on a
// miss).
template <bool kAny, class Stk>
__device__ __forceinline__ bool tri_traverse(const float4 *__restrict__ nodes,
                                             const float4 *__restrict__ prims,
                                             uint32_t max_nodes, uint32_t nprims,
                                             const RaySetup &s, bool ds, float kEPS,
                                             uint32_t prev, float tlimit, const Stk &st,
                                             float &t, float &u, float &v, uint32_t &prim) {
  const bool filter = kEPS >= 1e-30f;
  t = kAny ? tlimit : FLT_MAX;
  u = 0.0f;
  v = 0.0f;
  prim = SRF_NO_PRIM;
  int sp = 0;
  uint32_t cur = 0;
  uint4 meta;
  for (;;) {
    // descend until this lane holds a leaf (or has nothing left)
    for (;;) {
      if (cur >= max_nodes) {
        cur = kDone;
        break;
      }
      const float4 *nd = nodes + 4 * (size_t)cur;
      // the whole 64-byte node in one round trip (a leaf ignores the boxes)
      const float4 n0 = nd[0], n1 = nd[1], n2 = nd[2];
      meta = reinterpret_cast<const uint4 *>(nd)[3];
      keep_loaded(n0, n1, n2);
      if (meta.x != 0) break;
      const bool h0 = ray_aabb<true>(s, t, n0.x, n0.y, n0.z, n1.z, n1.w, n2.x);
      const bool h1 = ray_aabb<true>(s, t, n0.w, n1.x, n1.y, n2.y, n2.z, n2.w);
      const int nearc = (s.sbits >> meta.y) & 1u;
      const bool hn = nearc ? h1 : h0, hf = nearc ? h0 : h1;
      const uint32_t cn = nearc ? meta.w : meta.z, cf = nearc ? meta.z : meta.w;
      if (hn) {
        if (hf && sp < kTraceStack) st.put(sp++, cf);
        cur = cn;
      } else if (hf) {
        cur = cf;
      } else if (sp == 0) {
        cur = kDone;
        break;
      } else {
        cur = st.get(--sp);
      }
    }
    if (cur == kDone) break;
    // leaf: TestLeafNode, render/render_accel_triangle.cc:2386-2433; the
    // next triangle's 48 bytes are in flight while this one is tested
    const uint32_t first = meta.w, end = min(meta.w + meta.z, nprims);
    if (first < end) {
      const float4 *P = prims + 3 * (size_t)first;
      float4 A = P[0], B = P[1], C = P[2];
      for (uint32_t q = first; q < end; q++) {
        float4 nA = A, nB = B, nC = C;
        if (q + 1 < end) {
          P += 3;
          nA = P[0];
          nB = P[1];
          nC = P[2];
        }
        keep_loaded(nA, nB, nC);
        if (__float_as_uint(A.w) != prev) {
          float tt, uu, vv;
          if (tri_isect(s, A, B, C, ds, kEPS, filter, t, tt, uu, vv)) {
            if (kAny) {
              if (tt < tlimit) return true;
            } else {
              t = tt;
              u = uu;
              v = vv;
              prim = __float_as_uint(A.w);
            }
          }
        }
        A = nA;
        B = nB;
        C = nC;
      }
    }
    if (sp == 0) break;
    cur = st.get(--sp);
  }
  return false;
}

}  // namespace
}  // namespace srf
