// dtrace.h — two-level BVH traversal on the device.
//
// Per-lane DFS with the reference's visiting order, so that the winner of
// equal-t hits (t <= t_best accepts a later triangle, geometry/primitives.h:48)
// is the same triangle the CPU picks:
//   BLAS (geometry/blas.cpp:211-307): the root is not box-tested; interior
//     nodes pair-test both children with SSE MINPS/MAXPS semantics; closest
//     hit visits the child with the smaller entry distance first, ties visit
//     the right child first; any-hit visits the left child first.
//   TLAS (geometry/tlas.cpp:172-290): test-on-pop sign-selected slab test;
//     closest hit orders children by their box centres on the parent's
//     longest axis; instances transform the ray without normalising it so t
//     is shared by both spaces (geometry/transform.h:70-77).
//
// BLAS stack entries carry what the walk needs about a node without loading
// it: the node's child index and triangle count. The upload precomputes each
// node's entry into its record, so a pair test reads both children's entries
// with their boxes. Bits 28..31 hold the count (0 = interior: low bits = the
// left child of the pair; 1..14 = leaf: low bits = its first triangle slot;
// 15 = a leaf of 15 or more: low bits = its first slot, whose bigcnt word
// holds the count). Node and slot indices are < 2^28.
//
// Stack: the entry on top is held in a register (TravStack::tos). Of those
// below it the deepest `lds_depth` live in LDS, laid out entry-major
// ([entry][lane]) so lanes at equal depth hit distinct banks; the others
// spill, in order, to a per-lane HBM region. The BLAS walk of an instance
// runs on top of the TLAS entries, so both share kMaxStack; a marker entry
// (kEntEnd) under each BLAS walk ends it when it is popped.
#pragma once
#include "../common/dev_types.h"
#include "dmath.h"

namespace xnh {

// The kernels' dynamic LDS: lds_depth x blockDim.x stack entries.
extern __shared__ uint32_t trav_lds[];

constexpr uint32_t kEntEnd = kNoRoot;            // no entry: the lane is not in a BLAS walk
constexpr uint32_t kStackBottom = 0xFFFFFFFEu;   // the top of an empty stack (equals no entry)

struct TravStack {
  // LDS slots are byte addresses: an LDS pointer is 32 bits, and the walk
  // steps and compares them. They are signed: the row below a lane's first
  // slot lies below address 0 in a kernel whose LDS holds nothing else.
  typedef __attribute__((address_space(3))) uint32_t LdsWord;
  uint32_t tos;         // the entry on top (kStackBottom: the stack is empty)
  int32_t top;          // slot of the entry below it: bottom + row * (entries held)
  int32_t bottom;       // one row below this lane's first slot
  int32_t last;         // this lane's last slot (entries from lds_depth on are in the spill)
  uint32_t* spill;      // this lane's spill column: entry e is spill[(e - lds_depth) * spill_stride]
  int32_t row;          // bytes from one entry's slot to the next
  int spill_stride, lds_depth;   // lds_depth >= 1
  bool overflow;
  __device__ __forceinline__ void clear() {
    tos = kStackBottom;
    top = bottom;
  }
  __device__ __forceinline__ void reset() {
    clear();
    overflow = false;
  }
  __device__ __forceinline__ bool empty() const { return tos == kStackBottom; }
  __device__ __forceinline__ static LdsWord* word(int32_t slot) {
    return (LdsWord*)static_cast<uint32_t>(slot);
  }
  // Entries held (rarely needed: the walk compares slots instead).
  __device__ __forceinline__ int size() const { return static_cast<int>(static_cast<uint32_t>(top - bottom) / static_cast<uint32_t>(row)); }
  // The entry below the top, for a pop. The LDS read is issued for every
  // lane, at its last slot when the entry is in the spill, so that the walk
  // can issue it with its node loads; in_spill() lanes replace the value.
  __device__ __forceinline__ uint32_t below() const { return *word(min(top, last)); }
  __device__ __forceinline__ bool in_spill() const { return top > last; }
  __device__ __forceinline__ uint32_t spilled() const {
    return gld1(spill, static_cast<size_t>(size() - 1 - lds_depth) * static_cast<size_t>(spill_stride));
  }
  // Stores v, the former top, in the spill slot the stack has just grown
  // into (top was advanced). False past `limit` entries.
  __device__ __forceinline__ bool keep_spilled(uint32_t v, int limit) {
    const int n = size();
    if (n > limit) return false;
    gst1(spill, static_cast<size_t>(n - 1 - lds_depth) * static_cast<size_t>(spill_stride), v);
    return true;
  }
  // Entries beyond kMaxStack are not stored: the flag ends the ray. The
  // marker under a BLAS walk takes a place of its own (`extra`).
  __device__ __forceinline__ void push(uint32_t v, int extra = 0) {
    top += row;
    if (top <= last) {
      *word(top) = tos;
    } else if (!keep_spilled(tos, kMaxStack + extra)) {
      top -= row;
      overflow = true;
      return;
    }
    tos = v;
  }
  __device__ __forceinline__ uint32_t pop() {
    const uint32_t v = tos;
    tos = below();
    if (in_spill()) tos = spilled();
    top -= row;
    return v;
  }
};

// Traversal work counts. The rendering kernels have a counting variant
// (the same walk with these increments) used when work counts are asked
// for; the timed variant carries none of them.
struct TravCount {
  uint32_t node_tests, interior, tri_tests, inst_visits;
  // SIMD use: int_iters, leaf_iters and round_iters count wave iterations
  // (on one lane of the wave); leaf_steps and round_lanes count lanes
  uint32_t int_iters, leaf_iters, leaf_steps, round_iters, round_lanes;
};

// The lanes where p holds (as a lane mask, without the detour over an
// integer that HIP's __ballot takes), and how many.
__device__ __forceinline__ unsigned long long ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// (The empty asm keeps the count a 32-bit scalar; left to itself the compiler
// compares two such counts as 64-bit values on the vector unit.)
__device__ __forceinline__ int lanes_of(bool p) {
  int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(p));
  asm("" : "+s"(n));
  return n;
}

// True on the lowest active lane of the wave.
__device__ __forceinline__ bool first_active_lane() {
  return static_cast<int>(threadIdx.x & 63u) == __ffsll(static_cast<long long>(ballot(1))) - 1;
}

struct HitRef {
  float t, u, v;
  uint32_t slot;   // global leaf slot
  int32_t inst;    // instance index, -1 = none
};

struct TriRec {
  float4 a, b, c;
};
__device__ __forceinline__ TriRec load_tri(const float4* __restrict__ tris, uint32_t slot) {
  const size_t k = 3 * static_cast<size_t>(slot);
  return TriRec{gld4(tris, k), gld4(tris, k + 1), gld4(tris, k + 2)};
}

// Moller-Trumbore on a pre-gathered triangle (geometry/primitives.h:25-49).
// The reference's early returns are one conjunction here: lanes of a wave
// seldom fail together, so a branch per condition cost more than it skipped.
__device__ __forceinline__ bool tri_test(const TriRec& r, f3 o, f3 d, float tmin, float tmax, float& t, float& u,
                                         float& v) {
  const f3 v0{r.a.x, r.a.y, r.a.z}, e1{r.a.w, r.b.x, r.b.y}, e2{r.b.z, r.b.w, r.c.x};
  const f3 h = cross(d, e2);
  const float det = dot(e1, h);
  const float ia = 1.f / det;
  const f3 s = o - v0;
  u = ia * dot(s, h);
  const f3 q = cross(s, e1);
  v = ia * dot(d, q);
  t = ia * dot(e2, q);
  return !(fabsf(det) < 1e-7f) & !(u < 0.f) & !(u > 1.f) & !(v < 0.f) & !(u + v > 1.f) & (t >= tmin) & (t <= tmax);
}

// Two-child slab test: hits in hl/hr, near distances in tn0/tn1.
__device__ __forceinline__ void pair_test(float4 la, float4 lb, float4 ra, float4 rb, f3 inv, f3 o, float tmin,
                                          float tmax, float& tn0, float& tn1, bool& hl, bool& hr) {
  const float lx0 = (la.x - o.x) * inv.x, lx1 = (la.w - o.x) * inv.x;
  const float ly0 = (la.y - o.y) * inv.y, ly1 = (lb.x - o.y) * inv.y;
  const float lz0 = (la.z - o.z) * inv.z, lz1 = (lb.y - o.z) * inv.z;
  const float rx0 = (ra.x - o.x) * inv.x, rx1 = (ra.w - o.x) * inv.x;
  const float ry0 = (ra.y - o.y) * inv.y, ry1 = (rb.x - o.y) * inv.y;
  const float rz0 = (ra.z - o.z) * inv.z, rz1 = (rb.y - o.z) * inv.z;
  const float ln = xmax(xmax(xmax(xmin(lx0, lx1), xmin(ly0, ly1)), xmin(lz0, lz1)), tmin);
  const float lf = xmin(xmin(xmin(xmax(lx0, lx1), xmax(ly0, ly1)), xmax(lz0, lz1)), tmax);
  const float rn = xmax(xmax(xmax(xmin(rx0, rx1), xmin(ry0, ry1)), xmin(rz0, rz1)), tmin);
  const float rf = xmin(xmin(xmin(xmax(rx0, rx1), xmax(ry0, ry1)), xmax(rz0, rz1)), tmax);
  tn0 = ln;
  tn1 = rn;
  hl = ln <= lf;
  hr = rn <= rf;
}

// pair_test with the hardware min/max (v_min3/v_max3 chains instead of
// compare-and-select pairs). Equal to pair_test whenever no slab distance is
// NaN, and a NaN needs 0 * inf, so it is used only for rays whose origin,
// direction and inverse direction are finite in every component (box
// coordinates are finite). Without NaNs the two differ at
// most in the sign of a zero distance, which no comparison distinguishes.
__device__ __forceinline__ void pair_test_fast(float4 la, float4 lb, float4 ra, float4 rb, f3 inv, f3 o, float tmin,
                                               float tmax, float& tn0, float& tn1, bool& hl, bool& hr) {
  const float lx0 = (la.x - o.x) * inv.x, lx1 = (la.w - o.x) * inv.x;
  const float ly0 = (la.y - o.y) * inv.y, ly1 = (lb.x - o.y) * inv.y;
  const float lz0 = (la.z - o.z) * inv.z, lz1 = (lb.y - o.z) * inv.z;
  const float rx0 = (ra.x - o.x) * inv.x, rx1 = (ra.w - o.x) * inv.x;
  const float ry0 = (ra.y - o.y) * inv.y, ry1 = (rb.x - o.y) * inv.y;
  const float rz0 = (ra.z - o.z) * inv.z, rz1 = (rb.y - o.z) * inv.z;
  const float ln = fmaxf(fmaxf(fmaxf(fminf(lx0, lx1), fminf(ly0, ly1)), fminf(lz0, lz1)), tmin);
  const float lf = fminf(fminf(fminf(fmaxf(lx0, lx1), fmaxf(ly0, ly1)), fmaxf(lz0, lz1)), tmax);
  const float rn = fmaxf(fmaxf(fmaxf(fminf(rx0, rx1), fminf(ry0, ry1)), fminf(rz0, rz1)), tmin);
  const float rf = fminf(fminf(fminf(fmaxf(rx0, rx1), fmaxf(ry0, ry1)), fmaxf(rz0, rz1)), tmax);
  tn0 = ln;
  tn1 = rn;
  hl = ln <= lf;
  hr = rn <= rf;
}

__device__ __forceinline__ bool all_finite(f3 v) {
  return fabsf(v.x) < __builtin_huge_valf() && fabsf(v.y) < __builtin_huge_valf() &&
         fabsf(v.z) < __builtin_huge_valf();
}

// Written with selects rather than branches: it runs for both children of
// every interior step.
// Instance: world_to_local columns and metadata (see dev_types.h).
struct InstRec {
  f3 c0, c1, c2, c3;
  uint32_t root;
  int32_t id;
  uint32_t flat;       // the mesh has no vertex normals
  int32_t lmap;
};
__device__ __forceinline__ InstRec load_inst(const float4* inst, int i) {
  const float4 a = gld4(inst, 4 * i), b = gld4(inst, 4 * i + 1), c = gld4(inst, 4 * i + 2), m = gld4(inst, 4 * i + 3);
  InstRec r;
  r.c0 = f3{a.x, a.y, a.z};
  r.c1 = f3{a.w, b.x, b.y};
  r.c2 = f3{b.z, b.w, c.x};
  r.c3 = f3{c.y, c.z, c.w};
  r.root = __float_as_uint(m.x);
  r.id = __float_as_int(m.y);
  r.flat = __float_as_uint(m.z);
  r.lmap = __float_as_int(m.w);
  return r;
}

// ---- analytic primitives ------------------------------------------------------
// geometry/primitives.h:54-318 and geometry/prim_blas.cpp:165-229, with the
// reference's operation order (true divisions, std::min/std::max and the
// first-largest rule of std::max({...})).
struct PrimRec {
  int type, mat;
  float q[10];
};
__device__ __forceinline__ PrimRec load_prim(const float4* P, uint32_t i) {
  const float4 a = gld4(P, 3 * static_cast<size_t>(i)), b = gld4(P, 3 * static_cast<size_t>(i) + 1),
               c = gld4(P, 3 * static_cast<size_t>(i) + 2);
  PrimRec r;
  r.type = __float_as_int(a.x);
  r.mat = __float_as_int(a.y);
  r.q[0] = a.z; r.q[1] = a.w; r.q[2] = b.x; r.q[3] = b.y; r.q[4] = b.z;
  r.q[5] = b.w; r.q[6] = c.x; r.q[7] = c.y; r.q[8] = c.z; r.q[9] = c.w;
  return r;
}

// AABB::intersect (geometry/aabb.h:34-47) on a PrimBLAS node.
__device__ __forceinline__ bool prim_node_hit(float4 na, float4 nb, f3 o, f3 d, float rtmin, float rtmax,
                                              float& tnear) {
  const float tx0 = (na.x - o.x) / d.x, tx1 = (na.w - o.x) / d.x;
  const float ty0 = (na.y - o.y) / d.y, ty1 = (nb.x - o.y) / d.y;
  const float tz0 = (na.z - o.z) / d.z, tz1 = (nb.y - o.z) / d.z;
  float lo = smin(tx0, tx1), hi = smax(tx0, tx1);
  const float ly = smin(ty0, ty1), lz = smin(tz0, tz1), hy = smax(ty0, ty1), hz = smax(tz0, tz1);
  if (lo < ly) lo = ly;
  if (lo < lz) lo = lz;
  if (lo < rtmin) lo = rtmin;
  if (hy < hi) hi = hy;
  if (hz < hi) hi = hz;
  if (rtmax < hi) hi = rtmax;
  tnear = lo;
  return lo <= hi;
}

// Box slab walk (primitives.h:159-182): the entry distance and the entering
// face (axis, and whether it is the low face).
__device__ __forceinline__ bool prim_box_slabs(const PrimRec& p, f3 o, f3 d, float tmin, float rect, float& t,
                                               int& axis, bool& low) {
  const f3 c{p.q[0], p.q[1], p.q[2]}, h{p.q[3], p.q[4], p.q[5]};
  const f3 mn = c - h, mx = c + h;
  float t_lo = tmin, t_hi = rect;
  axis = 0;
  low = false;
  for (int i = 0; i < 3; ++i) {
    const float inv = 1.f / comp(d, i);
    float t0 = (comp(mn, i) - comp(o, i)) * inv;
    float t1 = (comp(mx, i) - comp(o, i)) * inv;
    const bool flip = inv < 0.f;
    if (flip) {
      const float tmp = t0;
      t0 = t1;
      t1 = tmp;
    }
    if (t0 > t_lo) {
      t_lo = t0;
      axis = i;
      low = !flip;
    }
    t_hi = smin(t_hi, t1);
    if (t_lo > t_hi) return false;
  }
  t = t_lo;
  return true;
}

// The primitive's intersect: a hit at t in [tmin, rect).
__device__ __forceinline__ bool prim_hit(const PrimRec& p, f3 o, f3 d, float tmin, float rect, float& t) {
  switch (p.type) {
    case 0: {   // sphere
      const f3 c{p.q[0], p.q[1], p.q[2]};
      const float r = p.q[3];
      const f3 oc = o - c;
      const float a = dot(d, d), hb = dot(oc, d), cc = dot(oc, oc) - r * r;
      const float disc = hb * hb - a * cc;
      if (disc < 0.f) return false;
      const float sq = sqrtf(disc);
      t = (-hb - sq) / a;
      if (t < tmin || t >= rect) {
        t = (-hb + sq) / a;
        if (t < tmin || t >= rect) return false;
      }
      return true;
    }
    case 1: {   // plane
      const f3 n{p.q[0], p.q[1], p.q[2]};
      const float denom = dot(n, d);
      if (fabsf(denom) < 1e-7f) return false;
      t = (p.q[3] - dot(n, o)) / denom;
      return !(t < tmin || t >= rect);
    }
    case 2: {   // box
      int axis;
      bool low;
      return prim_box_slabs(p, o, d, tmin, rect, t, axis, low);
    }
    case 3: {   // disk
      const f3 c{p.q[0], p.q[1], p.q[2]}, n{p.q[3], p.q[4], p.q[5]};
      const float denom = dot(n, d);
      if (fabsf(denom) < 1e-7f) return false;
      t = dot(c - o, n) / denom;
      if (t < tmin || t >= rect) return false;
      const f3 op = (o + t * d) - c;
      return !(dot(op, op) > p.q[6] * p.q[6]);
    }
    default: {   // quad
      const f3 org{p.q[0], p.q[1], p.q[2]}, u{p.q[3], p.q[4], p.q[5]}, v{p.q[6], p.q[7], p.q[8]};
      const f3 nr = cross(u, v);
      const float area_sq = dot(nr, nr);
      if (area_sq < 1e-14f) return false;
      const float denom = dot(nr, d);
      if (fabsf(denom) < 1e-9f) return false;
      t = dot(nr, org - o) / denom;
      if (t < tmin || t >= rect) return false;
      const f3 op = (o + t * d) - org;
      const float s = dot(cross(op, v), nr) / area_sq;
      const float tv = dot(cross(u, op), nr) / area_sq;
      return !(s < 0.f || s > 1.f || tv < 0.f || tv > 1.f);
    }
  }
}

// Normal (facing the ray) and (u, v) the primitive's intersect writes for a
// hit at t.
__device__ __forceinline__ f3 prim_normal(const PrimRec& p, f3 o, f3 d, float tmin, float t, float& u, float& v) {
  constexpr float kPi = 3.14159265358979323846f;
  constexpr float kInvPi = 1.f / kPi;
  const f3 pos = o + t * d;
  switch (p.type) {
    case 0: {
      const f3 c{p.q[0], p.q[1], p.q[2]};
      const f3 out = (pos - c) / p.q[3];
      const float phi = atan2f(-out.z, out.x) + kPi;
      const float theta = acosf(fminf(fmaxf(-out.y, -1.f), 1.f));
      u = phi * (0.5f * kInvPi);
      v = theta * kInvPi;
      return dot(out, d) < 0.f ? out : -out;
    }
    case 1: {
      const f3 n{p.q[0], p.q[1], p.q[2]};
      u = pos.x - floorf(pos.x);
      v = pos.z - floorf(pos.z);
      return dot(n, d) < 0.f ? n : -n;
    }
    case 2: {
      float tt;
      int axis;
      bool low;
      prim_box_slabs(p, o, d, tmin, __builtin_huge_valf(), tt, axis, low);
      f3 n{0.f, 0.f, 0.f};
      const float s = low ? -1.f : 1.f;
      if (axis == 0) n.x = s;
      else if (axis == 1) n.y = s;
      else n.z = s;
      if (dot(n, d) > 0.f) n = -n;
      const f3 c{p.q[0], p.q[1], p.q[2]}, h{p.q[3], p.q[4], p.q[5]};
      const f3 mn = c - h;
      const int ua = (axis + 1) % 3, va = (axis + 2) % 3;
      u = (comp(pos, ua) - comp(mn, ua)) / (2.f * comp(h, ua));
      v = (comp(pos, va) - comp(mn, va)) / (2.f * comp(h, va));
      return n;
    }
    case 3: {
      const f3 c{p.q[0], p.q[1], p.q[2]}, n{p.q[3], p.q[4], p.q[5]};
      const f3 op = pos - c;
      const f3 ref = fabsf(n.x) < 0.9f ? f3{1.f, 0.f, 0.f} : f3{0.f, 1.f, 0.f};
      const f3 tang = normalize(cross(n, ref));
      const f3 bita = cross(n, tang);
      float phi = atan2f(dot(op, bita), dot(op, tang));
      if (phi < 0.f) phi += 2.f * kPi;
      u = phi * (0.5f * kInvPi);
      v = sqrtf(dot(op, op)) / p.q[6];
      return dot(n, d) < 0.f ? n : -n;
    }
    default: {
      const f3 org{p.q[0], p.q[1], p.q[2]}, uu{p.q[3], p.q[4], p.q[5]}, vv{p.q[6], p.q[7], p.q[8]};
      const f3 nr = cross(uu, vv);
      const float area_sq = dot(nr, nr);
      const f3 op = pos - org;
      u = dot(cross(op, vv), nr) / area_sq;
      v = dot(cross(uu, op), nr) / area_sq;
      const f3 n = normalize(nr);
      return dot(nr, d) > 0.f ? -n : n;
    }
  }
}

// Scene walk as a resumable state machine, advanced one round at a time so
// a persistent kernel can retire a finished ray and start the next in the
// same lane while the rest of the wave keeps walking.
//
// A lane needs one of three kinds of step next: a TLAS step (no BLAS entry
// at hand), an interior step (test a node's two children, continue with the
// nearer hit one, push the farther) or a leaf step (test its triangles,
// continue with the entry on top of the stack). wave_step runs one kind at a
// time for the whole wave.
//
// What bounds it: instruction issue in large launches, the latency of a
// step's loads in small ones. The step loops therefore keep everything they
// decide on in a few registers: the entry at hand alone names the kind of
// step, the stack's top is a register and its slot a byte address, the entry
// below it is read with the node (a pop waits for nothing), a marker under
// each BLAS walk replaces the test for its end, and stack entries beyond the
// LDS part are handled in a branch that a wave takes only when one of its
// lanes needs it. Against a walk that held a reached leaf and its successor
// apart and branched on push, pop and spill per lane (about 90 vector and 80
// scalar instructions an interior step; 70 and 25 here): 1.3M-triangle mesh
// 1920x1080x256 302.5 -> 267.2 ms, 4096 instances 389.6 -> 364.5 ms, Cornell
// 512x512x64 15.1 -> 14.2 ms a pass.
//
// No step is taken early: a lane at a leaf walks no further interior
// nodes until the leaf is tested, since a node box tested against a t_best
// not yet lowered by the leaf's hits may let through a subtree the reference
// culls, and box and triangle rounding differ enough for such a subtree to
// hold a hit. Every box and triangle test therefore sees the reference's
// t_best, and results and work counts equal its recursive walk, ties
// included. Closest-hit rays follow the reference's visiting order: BLAS
// children nearer entry first, ties right first; TLAS
// children ordered by their centres (tlas.cpp:231-241); a TLAS leaf's instances
// (pushed in reverse) walked first to last. Any-hit rays
// take BLAS children farther first (the reference: left first,
// blas.cpp:303-304); the occlusion answer does not depend on the order, only
// the work does. Closest hit starts from t_best = +inf and
// ignores tmax, as Scene::intersect does with a default HitRecord; any hit
// uses [tmin, tmax]. A stack overflow ends the ray with what it has found.
__device__ __forceinline__ bool ent_interior(uint32_t e) { return e < (1u << kEntShift); }
__device__ __forceinline__ bool ent_leaf(uint32_t e) { return e - (1u << kEntShift) < kEntEnd - (1u << kEntShift); }

// The arrays of the interior and leaf steps, kept in scalar registers by the
// persistent kernels (the others are read from the job's record where they
// are used).
struct SceneTables {
  const float4* bnodes;
  const float4* tris;
  bool plain;   // tlas_plain
  __device__ __forceinline__ explicit SceneTables(const DevScene& S) : bnodes(S.bnodes), tris(S.tris), plain(S.tlas_plain != 0) {}
  __device__ __forceinline__ SceneTables() : bnodes(nullptr), tris(nullptr), plain(false) {}
};

// kPrims: the scene may hold analytic primitives (a variant, because their
// walk raises the register count of the whole kernel).
template <bool kAny, bool kCount = true, bool kPrims = true>
struct Walker {
  f3 o, d, inv;       // world ray
  f3 lo, ld, linv;    // instance-space ray of the BLAS walk in progress
  float tmin, tbest;
  float rtmax;        // the ray's tmax (bounds the primitives' box tests, aabb.h:43)
  int inst;           // instance of the BLAS walk
  uint32_t e;         // BLAS entry to process next (interior or leaf), kEntEnd outside a BLAS walk
  bool occluded;      // any hit: an occluder was found
  bool fast;          // lo, ld, linv finite: pair_test_fast is exact
  bool wfast;         // o, d, inv finite: no slab distance of a TLAS box is NaN (see node_step)
  HitRef hit;         // u, v, slot, inst of the closest hit; its t is tbest

  __device__ __forceinline__ void idle(TravStack& st) {
    e = kEntEnd;
    st.reset();
  }

  __device__ __forceinline__ void begin(const DevScene& S, f3 o_, f3 d_, float tmin_, float tmax_, TravStack& st,
                                        TravCount& c) {
    o = o_;
    d = d_;
    inv = f3{1.f / d.x, 1.f / d.y, 1.f / d.z};
    tmin = tmin_;
    rtmax = tmax_;
    tbest = kAny ? tmax_ : __builtin_huge_valf();
    inst = -1;
    e = kEntEnd;
    occluded = false;
    fast = false;
    hit = HitRef{0.f, 0.f, 0.f, 0u, -1};
    // the counting variant tests every node it pops, to count as the
    // reference does
    wfast = !kCount && all_finite(inv) && all_finite(d) && all_finite(o);
    st.reset();
    if (S.num_tnodes > 0) {
      if (kCount) ++c.node_tests;
      st.push(S.troot);
    }
  }

  __device__ __forceinline__ bool found() const { return kAny ? occluded : hit.inst >= 0; }

  // The walk is over: nothing on the stack, no BLAS entry at hand.
  __device__ __forceinline__ bool finished(const TravStack& st) const { return e == kEntEnd && st.empty(); }

  __device__ __forceinline__ void stop(TravStack& st) {
    e = kEntEnd;
    st.clear();
  }

  // The scene's primitives, walked to the end at once in the instance-space
  // ray lo/ld (PrimBLAS::intersect / ::intersects, prim_blas.cpp:165-229):
  // nodes tested when popped, children tested (closest hit) and pushed
  // nearer last; true when an any-hit walk found an occluder.
  __device__ __forceinline__ bool prim_walk(const DevScene& S, TravStack& st, TravCount& c) {
    if (S.num_pnodes <= 0) return false;
    const int32_t base = st.top;
    st.push(0u);
    while (st.top > base && !st.overflow) {
      const uint32_t idx = st.pop();
      const float4 na = gld4(S.pnodes, 2 * static_cast<size_t>(idx)), nb = gld4(S.pnodes, 2 * static_cast<size_t>(idx) + 1);
      float tn;
      if (kCount) ++c.node_tests;
      if (!prim_node_hit(na, nb, lo, ld, tmin, rtmax, tn)) continue;
      if (!kAny && tn > tbest) continue;
      const uint32_t child = __float_as_uint(nb.z), count = __float_as_uint(nb.w);
      if (count > 0) {
        for (uint32_t k = 0; k < count; ++k) {
          const uint32_t pi = gld1(S.porder, child + k);
          const PrimRec pr = load_prim(S.prims, pi);
          float t;
          if (kCount) ++c.tri_tests;
          if (prim_hit(pr, lo, ld, tmin, kAny ? rtmax : tbest, t)) {
            if (kAny) return true;   // the ray is finished
            tbest = t;
            hit.u = 0.f;
            hit.v = 0.f;
            hit.slot = pi | kPrimHit;
            hit.inst = inst;
          }
        }
        continue;
      }
      if (kAny) {
        st.push(child);
        st.push(child + 1);
        continue;
      }
      if (kCount) {
        ++c.interior;
        c.node_tests += 2;
      }
      float tl, tr;
      const bool hl = prim_node_hit(gld4(S.pnodes, 2 * static_cast<size_t>(child)),
                                    gld4(S.pnodes, 2 * static_cast<size_t>(child) + 1), lo, ld, tmin, rtmax, tl) &&
                      tl <= tbest;
      const bool hr = prim_node_hit(gld4(S.pnodes, 2 * static_cast<size_t>(child) + 2),
                                    gld4(S.pnodes, 2 * static_cast<size_t>(child) + 3), lo, ld, tmin, rtmax, tr) &&
                      tr <= tbest;
      if (hl && hr) {
        if (tl < tr) {
          st.push(child + 1);
          st.push(child);
        } else {
          st.push(child);
          st.push(child + 1);
        }
      } else if (hl) {
        st.push(child);
      } else if (hr) {
        st.push(child + 1);
      }
    }
    return false;
  }

  // Sign-selected slab test of a TLAS box against the world ray
  // (geometry/aabb.h:59-71): near and far planes by direction sign.
  // `plain` (a wfast ray, a box with lo <= hi): the smaller distance of an axis
  // is the near one (rounding is monotone), so the hardware's min and max
  // give the same answer in fewer instructions.
  __device__ __forceinline__ bool tlas_box(bool plain, float lx, float ly, float lz, float hx, float hy, float hz) const {
    if (!kCount && plain) {
      asm volatile("");   // (two branches, not one computation with selects)
      const float x0 = (lx - o.x) * inv.x, x1 = (hx - o.x) * inv.x;
      const float y0 = (ly - o.y) * inv.y, y1 = (hy - o.y) * inv.y;
      const float z0 = (lz - o.z) * inv.z, z1 = (hz - o.z) * inv.z;
      return fmaxf(fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fminf(z0, z1)), tmin) <=
             fminf(fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1)), tbest);
    }
    const bool sx = d.x < 0.f, sy = d.y < 0.f, sz = d.z < 0.f;
    const float txn = ((sx ? hx : lx) - o.x) * inv.x, txf = ((sx ? lx : hx) - o.x) * inv.x;
    const float tyn = ((sy ? hy : ly) - o.y) * inv.y, tyf = ((sy ? ly : hy) - o.y) * inv.y;
    const float tzn = ((sz ? hz : lz) - o.z) * inv.z, tzf = ((sz ? lz : hz) - o.z) * inv.z;
    const float lo_t = smax(smax(smax(tmin, txn), tyn), tzn);
    const float hi_t = smin(smin(smin(tbest, txf), tyf), tzf);
    return lo_t <= hi_t;
  }

  // The two kinds of TLAS step, by the entry on top of the stack (not empty).
  __device__ __forceinline__ static bool is_instance(uint32_t te) { return (te & kInstTag) != 0u; }

  // An instance: its BLAS walk starts (or the primitives are walked to the
  // end), if its leaf's box is hit at this time (kInstTest).
  __device__ __forceinline__ void instance_step(const DevScene& S, TravStack& st, TravCount& c, bool plain) {
    const uint32_t te = st.pop();
    const int ii = static_cast<int>(te & kInstIndexMask);
    const InstRec in = load_inst(S.inst, ii);
    const float4 ba = gld4(S.ibox, 2 * static_cast<size_t>(ii)), bb = gld4(S.ibox, 2 * static_cast<size_t>(ii) + 1);
    if (te >= kInstTest && !tlas_box(plain, ba.x, ba.y, ba.z, ba.w, bb.x, bb.y)) return;
    if (kCount) ++c.inst_visits;
    lo = in.c0 * o.x + in.c1 * o.y + in.c2 * o.z + in.c3;
    ld = in.c0 * d.x + in.c1 * d.y + in.c2 * d.z;
    linv = f3{1.f / ld.x, 1.f / ld.y, 1.f / ld.z};
    fast = all_finite(linv) && all_finite(ld) && all_finite(lo);
    inst = ii;
    if (in.root == kPrimRoot) {   // the primitives: walked here, to the end
      if (kPrims && prim_walk(S, st, c)) {
        occluded = true;
        stop(st);
      }
    } else if (in.root != kNoRoot) {   // (kNoRoot: an empty mesh)
      // the marker that ends the walk; at kMaxStack it is always taken
      st.push(kEntEnd, 1);
      e = in.root;
    }
    if (st.overflow) stop(st);
  }

  // A node. The reference tests a node's box when it pops the node, against
  // the t_best of that time, and pushes both children. Here both children
  // are tested when their parent is popped and only those hit are pushed,
  // and a popped interior node is not tested itself. The walk enters the
  // same instances at the same times:
  //   - t_best only falls, so a child that fails now fails when popped;
  //   - an instance's box is tested again when it is popped;
  //   - a popped interior node that t_best has meanwhile passed by pushes
  //     nothing: its children's slab distances are no nearer and no farther
  //     than its own (their boxes lie inside it, and subtraction of the same
  //     origin and multiplication by the same reciprocal round monotonically),
  //     so they fail too. This needs distances without NaN, and a direction
  //     of -0 or an origin on a plane of a flat box can make one; rays with
  //     a zero or non-finite component test the node first (wfast false).
  // A step per node hit instead of one per node tested (both children of
  // every node hit), and instances entered in steps of their own: 4096
  // instances 1920x1080x64 347 -> 219 ms a pass; with tlas_box's plain form
  // 211 -> 199.
  __device__ __forceinline__ void node_step(const DevScene& S, TravStack& st, TravCount& c, bool plain) {
    const uint32_t ni = st.pop();
    if ((kCount || !plain) && !wfast) {
      const float4 na = gld4(S.tnodes, 3 * static_cast<size_t>(ni)), nb = gld4(S.tnodes, 3 * static_cast<size_t>(ni) + 1);
      if (!tlas_box(false, na.x, na.y, na.z, na.w, nb.x, nb.y)) return;
    }
    const float4* rec = S.tpairs + 4 * static_cast<size_t>(ni);
    const float4 a = gld4(rec, 0), b = gld4(rec, 1), q = gld4(rec, 2), k = gld4(rec, 3);
    const uint32_t wl = __float_as_uint(k.z), right = __float_as_uint(k.w);
    const uint32_t ax = (wl >> kTlasAxisShift) & 3u;
    const bool hl = tlas_box(plain, a.x, a.y, a.z, a.w, b.x, b.y);
    if (ax == kTlasList) {   // a leaf of several instances (or one named twice): walked first to last
      if (hl)
        for (uint32_t n = __float_as_uint(b.z); n-- > 0u;) st.push(kInstTag | gld1(S.torder, right + n));
    } else {
      if (kCount) {
        ++c.interior;
        c.node_tests += 2;
      }
      const uint32_t left = wl & ~(3u << kTlasAxisShift);
      const bool hr = tlas_box(plain, b.z, b.w, q.x, q.y, q.z, q.w);
      const float oa = comp(o, static_cast<int>(ax)), ia = comp(inv, static_cast<int>(ax));
      const float tl = (k.x - oa) * ia;
      const float tr = (k.y - oa) * ia;
      const bool right_last = !kAny && tl < tr;   // any hit: left pushed first, as the reference does
      if (right_last ? hr : hl) st.push(right_last ? right : left);
      if (right_last ? hl : hr) st.push(right_last ? left : right);
    }
    if (st.overflow) stop(st);
  }

  // One interior step on e (an interior entry): pair-test its children,
  // continue with the nearer hit one, push the farther; with no child hit,
  // continue with the entry on top of the stack.
  template <bool kFast>
  __device__ __forceinline__ void interior_step(const SceneTables& T, TravStack& st, TravCount& c) {
    const float4* pair = T.bnodes + 2 * static_cast<size_t>(e);
    const float4 la = gld4(pair, 0), lb = gld4(pair, 1), ra = gld4(pair, 2), rb = gld4(pair, 3);
    const uint32_t below = st.below();
    float tn0, tn1;
    bool hl, hr;
    if (kCount) {
      ++c.interior;
      c.node_tests += 2;
    }
    if (kFast) pair_test_fast(la, lb, ra, rb, linv, lo, tmin, tbest, tn0, tn1, hl, hr);
    else pair_test(la, lb, ra, rb, linv, lo, tmin, tbest, tn0, tn1, hl, hr);
    const uint32_t el = __float_as_uint(lb.w), er = __float_as_uint(rb.w);
    // closest: nearer first, ties right first (blas.cpp:252-258). Any hit:
    // farther first. Occlusion does not depend on the order (every box is
    // tested against the fixed tmax); a shadow ray's nearer child is mostly
    // the box around its own origin, whose triangles it cannot hit, so the
    // farther child meets occluders sooner.
    const bool left_first = kAny ? !(tn0 < tn1) : tn0 < tn1;
    const bool both = hl && hr, none = !(hl || hr);
    const bool left = hl && (!hr || left_first);
    const uint32_t next = left ? el : er, other = left ? er : el;
    const uint32_t was = st.tos;
    const int32_t at = st.top, up = at + st.row;
    e = none ? was : next;
    st.tos = both ? other : (none ? below : was);
    st.top = both ? up : (none ? at - st.row : at);
    const bool fits = up <= st.last;
    if (both && fits) *TravStack::word(up) = was;
    // rare: lanes whose entry lies in the spill (one compare for the wave; the
    // camera rays' launches are bound by the vector unit, and a ballot of a
    // combined condition costs it two more instructions: with the plain
    // compares here and in interior_run k_camera took 42.8 -> 40.9 ms, k_trace
    // 126.6 -> 122.3, 1.3M-triangle mesh 1920x1080x256)
    if (ballot(up > st.last) != 0ull) {
      if (both && !fits) {
        if (!st.keep_spilled(was, kMaxStack + 1)) {
          st.overflow = true;
          stop(st);
        }
      } else if (none && at > st.last) {
        st.top = at;
        st.tos = st.spilled();
        st.top = at - st.row;
      }
    }
  }

  // Tests the leaf e and continues with the entry on top of the stack. The
  // first two triangles (a leaf of the reference's builder holds at most
  // two) are fetched together.
  __device__ __forceinline__ void leaf_step(const DevScene& S, const SceneTables& T, TravStack& st, TravCount& c) {
    uint32_t count = e >> kEntShift;
    const uint32_t first = e & kEntIndexMask;
    const TriRec r0 = load_tri(T.tris, first);
    const TriRec r1 = load_tri(T.tris, count > 1u ? first + 1u : first);
    const uint32_t below = st.below();
    bool ended = test_tri(r0, first, true, c);
    if (!kAny || !ended) ended = test_tri(r1, first + 1u, count > 1u, c);
    if (ballot(count > 2u) != 0ull) {   // larger leaves (equal centres, other builders)
      if (count == kEntBigLeaf) count = gld1(S.bigcnt, first);
      for (uint32_t k = 2; k < count && !(kAny && ended); ++k) ended = test_tri(load_tri(T.tris, first + k), first + k, true, c);
    }
    if (kAny && ended) {
      occluded = true;
      stop(st);
    } else {
      e = st.tos;
      st.tos = below;
      if (st.in_spill()) st.tos = st.spilled();
      st.top -= st.row;
    }
  }

  // Tests one triangle of the leaf (if `there`); a closest hit takes it, true
  // when an any-hit walk is done.
  __device__ __forceinline__ bool test_tri(const TriRec& r, uint32_t slot, bool there, TravCount& c) {
    float t, u, v;
    if (kCount && there) ++c.tri_tests;
    const bool yes = tri_test(r, lo, ld, tmin, tbest, t, u, v) && there;
    if (!kAny && yes) {
      tbest = t;   // the hit distance (hit.t is not kept during the walk)
      hit.u = u;
      hit.v = v;
      hit.slot = slot;
      hit.inst = inst;
    }
    return kAny && yes;
  }
};

// Interior steps of wave_step's lanes while interior steps keep the
// majority of the wave's BLAS lanes.
template <bool kFast, bool kAny, bool kCount, bool kPrims>
__device__ __forceinline__ void interior_run(Walker<kAny, kCount, kPrims>& w, const SceneTables& T, TravStack& st,
                                             TravCount& c) {
  int ni, nb;
  bool in = ent_interior(w.e);
  do {
    if (kCount && first_active_lane()) ++c.int_iters;
    if (in) w.template interior_step<kFast>(T, st, c);
    in = ent_interior(w.e);
    ni = lanes_of(in);
    nb = lanes_of(w.e < kEntEnd);   // interior and leaf (two plain compares)
  } while (ni != 0 && 2 * ni >= nb);
}

// TLAS steps of the nt lanes that need one, each in this run until it enters a
// BLAS or ends; each turn takes the kind, node or instance, that more of its
// lanes need.
template <bool kAny, bool kCount, bool kPrims>
__device__ __forceinline__ void tlas_run(Walker<kAny, kCount, kPrims>& w, const DevScene& S, TravStack& st,
                                         TravCount& c, int nt, bool plain) {
  bool part = w.e == kEntEnd && !st.empty();
  int n0 = nt;
  do {
    const bool instance = part && Walker<kAny, kCount, kPrims>::is_instance(st.tos);
    if (2 * lanes_of(instance) <= n0) {
      if (part && !instance) w.node_step(S, st, c, plain);
    } else {
      if (instance) w.instance_step(S, st, c, plain);
    }
    part = part && w.e == kEntEnd && !st.empty();
    n0 = lanes_of(part);
  } while (n0 != 0 && 2 * n0 >= nt);
}

// One scheduled run of a wave's walks. Every lane holding a ray names the
// kind of step it needs next (TLAS entry, leaf, or interior node pair);
// the kind most lanes need runs, on those lanes only, while the others wait:
// interior and leaf steps repeat while their kind keeps the majority of the
// wave's BLAS lanes, TLAS steps while at least half of the lanes that began
// the run still need one. Each lane's own steps still run one at a time in
// the reference's order, each seeing the t_best its earlier steps left:
// only the interleaving of different lanes' steps is chosen here, so results
// and work counts are the reference's. Scheduling by majority rather than
// letting every lane finish a whole descent before any leaf is tested keeps
// more lanes of each iteration busy (a wave's descents differ in length).
// Lanes without a ray (Walker::idle) and finished ones take no part. Runs
// follow each other until `rest` lanes take no part (the caller then gives
// them rays) or kTurns are done: going round the caller's loop between two
// runs cost as much as an interior step (Cornell 512x512x64 12.4 -> 12.0 ms,
// 1.3M-triangle mesh 1920x1080x256 240.7 -> 236.5 ms). With primitives, whose
// long instance steps leave lanes finished for longer, one run at a time
// (801x449x33 6.38 against 6.50 ms). Every lane of the wave must reach it.
// `plain`: the scene is tlas_plain and every lane with a ray wfast.
constexpr int kTurns = 64;
template <bool kAny, bool kCount, bool kPrims>
__device__ __forceinline__ void wave_step(Walker<kAny, kCount, kPrims>& w, const DevScene& S, const SceneTables& T,
                                          TravStack& st, TravCount& c, int rest, bool plain) {
  for (int turn = 0; turn < (kPrims ? 1 : kTurns); ++turn) {
    const int nt = lanes_of(w.e == kEntEnd && !st.empty());
    int ni = lanes_of(ent_interior(w.e)), nl = lanes_of(w.e < kEntEnd) - ni;
    if (64 - (nt + nl + ni) >= rest && turn > 0) return;
    if (ni >= nl && ni >= nt) {
      // the hardware min/max slab test when every walking lane's ray allows it
      // (a wave-uniform choice). The two runs are separate loops: with one
      // loop and the choice inside it, the compiler computed the slab
      // distances before the branch, and the min/max instructions then
      // re-canonicalised each of them (a value from another block may be a
      // signalling NaN), 12 more instructions per node pair.
      if (ni == 0) return;
      if (ballot(ent_interior(w.e) && !w.fast) == 0ull) interior_run<true>(w, T, st, c);
      else interior_run<false>(w, T, st, c);
    } else if (nl >= nt) {
      do {
        if (kCount && first_active_lane()) ++c.leaf_iters;
        if (ent_leaf(w.e)) {
          if (kCount) ++c.leaf_steps;
          w.leaf_step(S, T, st, c);
        }
        ni = lanes_of(ent_interior(w.e));
        nl = lanes_of(w.e < kEntEnd) - ni;
      } while (nl != 0 && nl >= ni);
    } else {
      tlas_run(w, S, st, c, nt, plain);
    }
  }
}

// Whole walk of one ray per lane (the ray-batch API), with work counts.
// Every lane of the wave must reach it.
template <bool kAny>
__device__ __forceinline__ bool walk_scene(const DevScene& S, f3 o, f3 d, float tmin, float tmax, bool valid,
                                           HitRef& hit, TravStack& st, TravCount& c) {
  Walker<kAny> w;
  const SceneTables T(S);
  w.begin(S, o, d, tmin, tmax, st, c);
  if (!valid) w.stop(st);
  const bool plain = T.plain && ballot(!w.wfast) == 0ull;
  for (uint32_t guard = 0; ballot(!w.finished(st)) != 0ull; ++guard) {
    if (guard >= kWaveStepLimit) {
      st.overflow = true;
      break;
    }
    wave_step(w, S, T, st, c, 64, plain);
  }
  hit = w.hit;
  hit.t = w.found() ? w.tbest : 0.f;
  return valid && w.found();
}

}  // namespace xnh
