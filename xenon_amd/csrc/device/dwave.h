// dwave.h — wave-level helpers and batch bookkeeping shared by the
// wavefront kernels (kernels.hip) and the guided-rendering kernels
// (guide.hip): ballot compaction, wave reductions, traversal-counter
// flushes, the per-block view of the current batch's chunk table, and the
// surface record of a closest hit.
#pragma once
#include <hip/hip_runtime.h>

#include "../common/dev_types.h"
#include "dmath.h"
#include "dtrace.h"

namespace xnh {

constexpr float kBounceOffset = 1e-4f;   // math/ray.h:13
constexpr float kShadowOff = 5e-4f;      // math/ray.h:14

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x & 63u); }

// The job table is written by the host before a batch and is read-only while
// kernels run. Read through the constant address space at a wave-uniform
// index, a job's fields are scalar loads (the scalar cache, counted by
// lgkmcnt). As generic loads inside divergent code they were per-lane vector
// loads, each a round trip before the array it names could be read, and each
// wait for one also waited for the wave's pending stores (vmcnt counts both).
// The returned references are generic aliases of the constant-space object;
// once inlined, the compiler infers the address space of the loads through
// them. (A copy by value was kept in scratch memory.) The host compilation
// pass parses these bodies but never runs them; the cast exists only for the
// device.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const DevJob ConstJob;
__device__ __forceinline__ const DevJob& job_rec(const DevJob* jobs, int job) {
  return reinterpret_cast<const ConstJob*>(reinterpret_cast<uintptr_t>(jobs))[job];
}
#else
__device__ __forceinline__ const DevJob& job_rec(const DevJob* jobs, int job) { return jobs[job]; }
#endif
__device__ __forceinline__ const DevScene& job_scene(const DevJob* jobs, int job) { return job_rec(jobs, job).S; }

// A batch's paths are laid out in 8x8 pixel tiles, so that the 64 primary
// rays of a wave leave one compact patch of the image (a 64x1 row strip
// spreads over eight times the width): the image is cut into bands of 8 rows
// (the last band may be lower), a band into blocks of 8 columns (the last
// block may be narrower), and a block is enumerated row by row. Maps the
// tiled index t in [0, W*H) to the pixel index y*W + x (a bijection).
__device__ __forceinline__ int tiled_pixel(int t, int W, int H) {
  const int band = t / (8 * W);
  const int r = t - band * 8 * W;
  const int hb = min(8, H - 8 * band);
  const int bx = r / (8 * hb);
  const int wb = min(8, W - 8 * bx);
  const int q = r - bx * 8 * hb;
  const int yi = q / wb;
  return (8 * band + yi) * W + 8 * bx + (q - yi * wb);
}

// The camera path behind depth-0 queue entry e of chunk ck: depth 0 holds a
// chunk's paths as its segment 0. Slots are sample-major over the tiled
// pixels (slot = base + sample * npix + t, t the tiled pixel index). The
// entries are in slot order, or, when ck.cam_lg = lg is set, in blocks of
// 64: 2^lg samples of 2^(6-lg) consecutive tiled pixels (lg 3: a row of an
// 8x8 tile; lg 6: one pixel), block after block over the pixels, then over
// the next 2^lg samples, so that a wave's camera rays leave a footprint
// 2^lg times smaller than a tile, while each sample's 2^(6-lg) slots stay
// contiguous (2^lg divides the chunk's samples, 2^(6-lg) its pixels). Its
// seed is the pixel index plus the
// sample index times 0xdeadbeef, its ray the jittered pinhole ray
// (cpu_tiled.cpp:20-29, camera/camera.h:35-37), and rng is the state after
// the two jitter draws. Camera rays are not stored: the depth-0 traversal,
// shading and guide inference each rebuild them here from the entry index,
// bit for bit the same wherever they are made.
struct CameraPath {
  f3 o, d;
  Rng rng;
  uint32_t slot;
};
__device__ __forceinline__ uint32_t fdiv(uint32_t n, FastDiv f) {
  return static_cast<uint32_t>((static_cast<uint64_t>(n) * f.m) >> f.p);
}
__device__ __forceinline__ CameraPath camera_path(const DevChunk& ck, const DevJob& J, uint32_t e) {
  // the divisions by the chunk's and the job's sizes are multiply-shifts
  // (FastDiv); the rest are shifts except in the last tile row and column
  const uint32_t local = e - static_cast<uint32_t>(ck.qbase);
  const uint32_t npix = static_cast<uint32_t>(ck.npix);
  uint32_t s, t;
  if (ck.cam_lg) {
    const uint32_t lg = static_cast<uint32_t>(ck.cam_lg), lp = 6u - lg;   // log2 of the samples, pixels per block
    const uint32_t blk = local >> 6, l = local & 63u;
    const uint32_t sg = fdiv(blk, ck.sdiv);   // / (npix >> lp)
    s = (sg << lg) + (l >> lp);
    t = ((blk - sg * (npix >> lp)) << lp) + (l & ((1u << lp) - 1u));
  } else {
    s = fdiv(local, ck.sdiv);   // / npix
    t = local - s * npix;
  }
  // tiled index -> pixel (x, y): the steps of tiled_pixel
  const int W = J.W, H = J.H;
  const int ti = static_cast<int>(t);
  const int band = static_cast<int>(fdiv(t, J.band));   // / (8 W)
  const int r = ti - band * 8 * W;
  const int hb = min(8, H - 8 * band);
  const int bx = hb == 8 ? r >> 6 : r / (8 * hb);
  const int wb = min(8, W - 8 * bx);
  const int q = r - bx * 8 * hb;
  const int yi = wb == 8 ? q >> 3 : q / wb;
  const int x = 8 * bx + (q - yi * wb), y = 8 * band + yi;
  const int pixel = y * W + x;
  const int spp = ck.spp_first + static_cast<int>(s);
  const uint64_t seed = static_cast<uint64_t>(pixel) + static_cast<uint64_t>(spp) * 0xdeadbeefULL;
  CameraPath p;
  p.rng = rng_for(seed);
  const float fx = static_cast<float>(x) + p.rng.f();
  const float fy = static_cast<float>(y) + p.rng.f();
  const float u = fx / static_cast<float>(J.W), w = fy / static_cast<float>(J.H);
  p.o = f3{J.cam.eye[0], J.cam.eye[1], J.cam.eye[2]};
  const f3 llc{J.cam.llc[0], J.cam.llc[1], J.cam.llc[2]};
  const f3 hz{J.cam.horiz[0], J.cam.horiz[1], J.cam.horiz[2]};
  const f3 vt{J.cam.vert[0], J.cam.vert[1], J.cam.vert[2]};
  p.d = normalize(llc + u * hz + w * vt - p.o);
  p.slot = static_cast<uint32_t>(ck.base) + s * npix + t;
  return p;
}

// Wave-aggregated append: one atomic per wave, ranks by ballot prefix.
// Must be reached by every lane of the wave.
__device__ __forceinline__ uint32_t wave_append(uint32_t* ctr, bool want) {
  const unsigned long long mask = __ballot(want);
  if (mask == 0ull) return 0u;
  const int lane = lane_id();
  const uint32_t rank = static_cast<uint32_t>(__popcll(mask & ((1ull << lane) - 1ull)));
  const int leader = __ffsll(static_cast<long long>(mask)) - 1;
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(ctr, static_cast<uint32_t>(__popcll(mask)));
  base = __shfl(base, leader);
  return base + rank;
}

// Two appends to one counter with one atomic: the `a` lanes take the first
// popcount(a) places of the wave's block, the `b` lanes the places after
// them. Must be reached by every lane of the wave.
__device__ __forceinline__ void wave_append2(uint32_t* ctr, bool a, bool b, uint32_t& ia, uint32_t& ib) {
  const unsigned long long ma = __ballot(a);
  const unsigned long long mb = __ballot(b);
  ia = ib = 0u;
  if ((ma | mb) == 0ull) return;
  const int lane = lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  const uint32_t na = static_cast<uint32_t>(__popcll(ma));
  const int leader = __ffsll(static_cast<long long>(ma | mb)) - 1;
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(ctr, na + static_cast<uint32_t>(__popcll(mb)));
  base = __shfl(base, leader);
  ia = base + static_cast<uint32_t>(__popcll(ma & below));
  ib = base + na + static_cast<uint32_t>(__popcll(mb & below));
}

// The shading kernel's appends of one pass: shadow records (the `a` lanes,
// then the `b` lanes) to ctr_s and continuations (`c` lanes) to ctr_c. The
// leader issues both atomics before either result is read, so their round
// trips overlap (one after the other, the second atomic's wait had cost as
// much as the rest of the pass). Must be reached by every lane of the wave.
__device__ __forceinline__ void wave_append_pass(uint32_t* ctr_s, bool a, bool b, uint32_t& ia, uint32_t& ib,
                                                 uint32_t* ctr_c, bool c, uint32_t& ic) {
  const unsigned long long ma = __ballot(a), mb = __ballot(b), mc = __ballot(c);
  ia = ib = ic = 0u;
  if ((ma | mb | mc) == 0ull) return;
  const int lane = lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  const uint32_t na = static_cast<uint32_t>(__popcll(ma));
  const uint32_t ns = na + static_cast<uint32_t>(__popcll(mb)), nc = static_cast<uint32_t>(__popcll(mc));
  const int leader = __ffsll(static_cast<long long>(ma | mb | mc)) - 1;
  uint32_t bs = 0u, bc = 0u;
  if (lane == leader) {
    if (ns) bs = atomicAdd(ctr_s, ns);
    if (nc) bc = atomicAdd(ctr_c, nc);
  }
  // one broadcast of both results: the wait for either comes after both
  // atomics are issued
  const unsigned long long both =
      __shfl(static_cast<unsigned long long>(bc) << 32 | static_cast<unsigned long long>(bs), leader);
  bs = static_cast<uint32_t>(both);
  bc = static_cast<uint32_t>(both >> 32);
  ia = bs + static_cast<uint32_t>(__popcll(ma & below));
  ib = bs + na + static_cast<uint32_t>(__popcll(mb & below));
  ic = bc + static_cast<uint32_t>(__popcll(mc & below));
}

__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Wave-reduced ray and (with `work`) traversal counters; `any` selects the
// shadow slots.
__device__ __forceinline__ void flush_counts(unsigned long long* stats, const TravCount& c, uint32_t rays, bool any,
                                             bool work = true) {
  const unsigned long long r = wave_sum(rays);
  if (lane_id() == 0 && r) atomicAdd(&stats[any ? kStShadow : kStClosest], r);
  if (!work) return;
  const unsigned long long a = wave_sum(c.node_tests), b = wave_sum(c.interior), t = wave_sum(c.tri_tests),
                           i = wave_sum(c.inst_visits);
  const int base = any ? kStShNodeTests : kStNodeTests;
  if (lane_id() == 0) {
    if (a) atomicAdd(&stats[base], a);
    if (b) atomicAdd(&stats[base + 1], b);
    if (t) atomicAdd(&stats[base + 2], t);
    if (i) atomicAdd(&stats[base + 3], i);
  }
  const unsigned long long p[5] = {wave_sum(c.int_iters), wave_sum(c.leaf_iters), wave_sum(c.leaf_steps),
                                   wave_sum(c.round_iters), wave_sum(c.round_lanes)};
  const int pbase = any ? kStShIntIters : kStIntIters;
  if (lane_id() == 0)
    for (int k = 0; k < 5; ++k)
      if (p[k]) atomicAdd(&stats[pbase + k], p[k]);
}

__device__ __forceinline__ TravStack make_stack(uint32_t* spill, int lds_depth) {
  TravStack st;
  // the dynamic LDS's byte address (its low 32 bits as a generic pointer)
  const int32_t base = static_cast<int32_t>(reinterpret_cast<uintptr_t>((TravStack::LdsWord*)trav_lds));
  st.row = static_cast<int32_t>(4u * blockDim.x);
  st.bottom = base + static_cast<int32_t>(4u * threadIdx.x) - st.row;
  st.last = st.bottom + lds_depth * st.row;
  st.spill = spill + (static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x);
  st.spill_stride = static_cast<int>(gridDim.x * blockDim.x);
  st.lds_depth = lds_depth;
  st.reset();
  return st;
}

// Surface data of a closest hit: the reference's HitRecord after
// intersect_triangle (geometry/mesh.h:104-129) and TLAS::fixup_hit
// (geometry/tlas.cpp:156-168).
struct Surface {
  f3 pos, n, gn;
  int mat;
  uint32_t tri;
  int32_t inst_id;
  int32_t lmap;
  bool front;
};

__device__ __forceinline__ f3 normal_out(const InstRec& in, f3 n) {
  return normalize(f3{in.c0.x * n.x + in.c0.y * n.y + in.c0.z * n.z, in.c1.x * n.x + in.c1.y * n.y + in.c1.z * n.z,
                      in.c2.x * n.x + in.c2.y * n.y + in.c2.z * n.z});
}

// A primitive hit: the primitive's own normal (facing the ray) and uv in
// instance space, then TLAS::fixup_hit (tlas.cpp:156-168).
__device__ __forceinline__ Surface resolve_prim(const DevScene& S, const HitRef& h, const InstRec& in, f3 o, f3 d,
                                               float tmin, float& u, float& v) {
  const uint32_t pi = h.slot & ~kPrimHit;
  const PrimRec pr = load_prim(S.prims, pi);
  const f3 lo = in.c0 * o.x + in.c1 * o.y + in.c2 * o.z + in.c3;
  const f3 ld = in.c0 * d.x + in.c1 * d.y + in.c2 * d.z;
  const f3 nl = prim_normal(pr, lo, ld, tmin, h.t, u, v);
  Surface s;
  s.tri = pi;
  s.pos = o + h.t * d;
  s.n = normal_out(in, nl);
  s.gn = s.n;
  s.front = dot(s.gn, d) < 0.f;
  s.mat = pr.mat;
  s.inst_id = in.id;
  s.lmap = -1;
  return s;
}

__device__ __forceinline__ Surface resolve(const DevScene& S, const HitRef& h, f3 o, f3 d, float tmin = 0.f) {
  const InstRec in = load_inst(S.inst, h.inst);
  if (h.slot & kPrimHit) {
    float u, v;
    return resolve_prim(S, h, in, o, d, tmin, u, v);
  }
  const float4* rec = S.tris + 3 * static_cast<size_t>(h.slot);
  const float4 a = rec[0], b = rec[1], c = rec[2];
  const int4 ts = S.tsurf[h.slot];
  const f3 e1{a.w, b.x, b.y}, e2{b.z, b.w, c.x};
  Surface s;
  s.tri = __float_as_uint(c.y);
  const f3 gl = normalize(cross(e1, e2));
  f3 nl = gl;
  if (!in.flat) {
    const f3 n0 = xyz(S.vnrm[ts.x]), n1 = xyz(S.vnrm[ts.y]), n2 = xyz(S.vnrm[ts.z]);
    nl = normalize(n0 * (1.f - h.u - h.v) + n1 * h.u + n2 * h.v);
  }
  s.pos = o + h.t * d;
  s.n = normal_out(in, nl);
  s.gn = normal_out(in, gl);
  s.front = dot(s.gn, d) < 0.f;
  s.mat = ts.w;
  s.inst_id = in.id;
  s.lmap = in.lmap;
  return s;
}

// The part of `resolve` the guide needs: position, world geometric normal,
// material and the light-map lookup of the hit triangle.
struct GeoSurface {
  f3 pos, gn;
  int mat;
  uint32_t tri;
  int32_t lmap;
};

__device__ __forceinline__ GeoSurface resolve_geo(const DevScene& S, const HitRef& h, f3 o, f3 d, float tmin = 0.f) {
  const InstRec in = load_inst(S.inst, h.inst);
  if (h.slot & kPrimHit) {
    float u, v;
    const Surface f = resolve_prim(S, h, in, o, d, tmin, u, v);
    return GeoSurface{f.pos, f.gn, f.mat, f.tri, -1};
  }
  const float4* rec = S.tris + 3 * static_cast<size_t>(h.slot);
  const float4 a = rec[0], b = rec[1], c = rec[2];
  const int4 ts = S.tsurf[h.slot];
  const f3 e1{a.w, b.x, b.y}, e2{b.z, b.w, c.x};
  GeoSurface s;
  s.tri = __float_as_uint(c.y);
  s.pos = o + h.t * d;
  s.gn = normal_out(in, normalize(cross(e1, e2)));
  s.mat = ts.w;
  s.lmap = in.lmap;
  return s;
}

// Gradient sky (scene/environment.h:34-46).
__device__ __forceinline__ f3 sky_eval(const DevSky& k, f3 d) {
  const f3 hz{k.horizon[0], k.horizon[1], k.horizon[2]};
  if (d.y < 0.f) {
    const float t = smin(-d.y, 1.f);
    return k.intensity * lerp3(hz, f3{k.ground[0], k.ground[1], k.ground[2]}, t);
  }
  const float t = pow_r(d.y, 1.0f / k.sharpness);
  return k.intensity * lerp3(hz, f3{k.zenith[0], k.zenith[1], k.zenith[2]}, t);
}


// ---- batch bookkeeping ------------------------------------------------------

// Per-block copy of the current batch's chunk table with the entry count of
// every queue segment and prefix sums of 64-entry work units over chunks
// (traversal / shading) or of pixels (accumulation).
struct BatchView {
  int batch, nch;
  DevChunk ch[kMaxChunks];
  uint32_t cnt[kMaxChunks][kQSeg];
  uint32_t prefix[kMaxChunks + 1];
};

// One queue's view in the traversal kernels: its segments' entry counts and
// the prefix sums of units over chunks.
struct TraceQueue {
  uint32_t cnt[kMaxChunks][kQSeg];
  uint32_t prefix[kMaxChunks + 1];
};
struct TraceChunk {
  int32_t job, qbase, qseg;
};
// What the traversal of bounce and shadow rays needs of the batch.
struct TraceView {
  int nch;
  uint32_t batch_units;   // units of the batch at depth 0
  TraceChunk ch[kMaxChunks];
  TraceQueue q[2];        // the path queue, the shadow queue
};
// A queue as find_chunk, unit_segment and trace_queue take it (a BatchView
// has the same members).
struct TraceUnits {
  const int& nch;
  const TraceChunk* ch;
  const uint32_t (*cnt)[kQSeg];
  const uint32_t* prefix;
  __device__ __forceinline__ TraceUnits(const TraceView& v, int q)
      : nch(v.nch), ch(v.ch), cnt(v.q[q].cnt), prefix(v.q[q].prefix) {}
};

// A queue's segment counts. counts: its counter of chunk 0, segment 0, as
// ctr_path / ctr_shadow give it, with mul 1 (path queue) or 2 (shadow
// queue). A count is clamped to its segment (segment 0 of a path queue may
// hold the chunk's whole region: depth 0), so reads stay inside the chunk's
// region even if an append ever overflowed a segment.
template <class Chunk>
__device__ __forceinline__ void load_counts(uint32_t (*cnt)[kQSeg], const Chunk* ch, int nch, const uint32_t* counts,
                                            uint32_t mul) {
  for (int t = static_cast<int>(threadIdx.x); t < nch * kQSeg; t += static_cast<int>(blockDim.x)) {
    const int ci = t / kQSeg, x = t % kQSeg;
    const uint32_t qseg = static_cast<uint32_t>(ch[ci].qseg);
    const uint32_t room = mul * ((mul == 1u && x == 0) ? static_cast<uint32_t>(kQSeg) * qseg : qseg);
    cnt[ci][x] = counts ? min(counts[t * kCtrStride], room) : 0u;
  }
}
__device__ __forceinline__ uint32_t chunk_units(const uint32_t (*cnt)[kQSeg], int ci) {
  uint32_t acc = 0;
  for (int x = 0; x < kQSeg; ++x) acc += (cnt[ci][x] + 63u) >> 6;
  return acc;
}
// Prefix sums over chunks by the work-group's first wave, lane t holding
// chunk t's `acc` (a scan: one thread adding up 64 chunks' counts took 10 us
// of each launch).
__device__ __forceinline__ void scan_chunks(uint32_t* prefix, uint32_t acc, int nch) {
  static_assert(kMaxChunks == 64, "one lane per chunk");
  const int lane = static_cast<int>(threadIdx.x);
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(acc, o);
    if (lane >= o) acc += t;
  }
  if (lane == 0) prefix[0] = 0u;
  if (lane < nch) prefix[lane + 1] = acc;
}

// Loads the batch and builds prefix[] from the segment counts (see
// load_counts), or, with counts null, over pixels. Every work-group of every
// launch starts with it, so its dependent loads are few: batch index, then
// the chunks and their number, then the counts. Block-wide; ends with a
// barrier.
__device__ __forceinline__ void load_batch(BatchView& v, const WaveBuffers& B, const uint32_t* counts, bool pixels) {
  const int tid = static_cast<int>(threadIdx.x);
  const int batch = static_cast<int>(B.counters[kBatch]);
  const int nch = B.nchunks[batch];
  if (tid == 0) {
    v.batch = batch;
    v.nch = nch;
  }
  if (tid < nch) v.ch[tid] = B.chunks[batch * kMaxChunks + tid];
  __syncthreads();
  if (counts) {
    load_counts(v.cnt, v.ch, nch, counts, 1u);
    __syncthreads();
  }
  if (tid < 64) {
    uint32_t acc = 0;
    if (tid < nch) acc = pixels ? static_cast<uint32_t>(v.ch[tid].npix) : chunk_units(v.cnt, tid);
    scan_chunks(v.prefix, acc, nch);
  }
  __syncthreads();
}

// The same for the traversal of a path queue (counts) and a shadow queue
// (shadow_counts); either may be null: no units of it.
__device__ __forceinline__ void load_trace(TraceView& v, const WaveBuffers& B, const uint32_t* counts,
                                           const uint32_t* shadow_counts) {
  const int tid = static_cast<int>(threadIdx.x);
  const int batch = static_cast<int>(B.counters[kBatch]);
  const int nch = B.nchunks[batch];
  if (tid < nch) {
    const DevChunk& ck = B.chunks[batch * kMaxChunks + tid];
    v.ch[tid] = TraceChunk{ck.job, ck.qbase, ck.qseg};
    if (tid == nch - 1) v.batch_units = static_cast<uint32_t>(ck.base + ck.cap) >> 6;
  }
  if (tid == 0) {
    v.nch = nch;
    if (nch == 0) v.batch_units = 0u;
  }
  __syncthreads();
  load_counts(v.q[0].cnt, v.ch, nch, counts, 1u);
  load_counts(v.q[1].cnt, v.ch, nch, shadow_counts, 2u);
  __syncthreads();
  if (tid < 64)
    for (int k = 0; k < 2; ++k) scan_chunks(v.q[k].prefix, tid < nch ? chunk_units(v.q[k].cnt, tid) : 0u, nch);
  __syncthreads();
}

// The persistent traversal kernels' counts. Every entry of the launch's queue
// is one ray, so without work counters the first work-group adds the queue's
// length (every work-group adding its own rays was a thousand atomics on one
// address at the end of each launch). The counting variants sum over the
// work-group and add with one atomic per counter and work-group; every
// thread of the work-group must reach it (256 threads). `any` selects the
// shadow slots.
template <bool kWork>
__device__ __forceinline__ void flush_counts_block(unsigned long long* stats, const uint32_t (*cnt)[kQSeg], int nch,
                                                   const TravCount& c, uint32_t rays, bool any) {
  if constexpr (!kWork) {
    if (blockIdx.x == 0 && threadIdx.x < 64u) {
      unsigned long long n = 0;
      if (static_cast<int>(threadIdx.x) < nch)
        for (int x = 0; x < kQSeg; ++x) n += cnt[threadIdx.x][x];
      n = wave_sum(n);
      if (threadIdx.x == 0 && n) atomicAdd(&stats[any ? kStShadow : kStClosest], n);
    }
  } else {
    constexpr int kN = 10;
    __shared__ unsigned long long red[kN][256 / 64];
    const int w = static_cast<int>(threadIdx.x >> 6), nw = static_cast<int>(blockDim.x >> 6);
    const unsigned long long n[kN] = {
        wave_sum(rays),         wave_sum(c.node_tests), wave_sum(c.interior),    wave_sum(c.tri_tests),
        wave_sum(c.inst_visits), wave_sum(c.int_iters),  wave_sum(c.leaf_iters),  wave_sum(c.leaf_steps),
        wave_sum(c.round_iters), wave_sum(c.round_lanes)};
    if (lane_id() == 0)
      for (int k = 0; k < kN; ++k) red[k][w] = n[k];
    __syncthreads();
    if (threadIdx.x < static_cast<unsigned>(kN)) {
      unsigned long long t = 0;
      for (int k = 0; k < nw; ++k) t += red[threadIdx.x][k];
      const int k = static_cast<int>(threadIdx.x);
      int slot;
      if (k == 0) slot = any ? kStShadow : kStClosest;
      else if (k < 5) slot = (any ? kStShNodeTests : kStNodeTests) + k - 1;
      else slot = (any ? kStShIntIters : kStIntIters) + k - 5;
      if (t) atomicAdd(&stats[slot], t);
    }
    __syncthreads();   // red may be written again
  }
}

// Slot `slot` of a per-slot radiance array.
__device__ __forceinline__ f3 slot_f3(const float* a, uint32_t slot) {
  const float* p = a + 3 * static_cast<size_t>(slot);
  return f3{p[0], p[1], p[2]};
}
__device__ __forceinline__ void put_slot(float* a, uint32_t slot, f3 v) {
  float* p = a + 3 * static_cast<size_t>(slot);
  p[0] = v.x;
  p[1] = v.y;
  p[2] = v.z;
}

// Last chunk c with prefix[c] <= u: the (non-empty) chunk holding item u.
template <class View>
__device__ __forceinline__ int find_chunk(const View& v, uint32_t u) {
  int lo = 0, hi = v.nch;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (v.prefix[mid] <= u) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Unit uc of chunk ci's units (segment by segment): returns the queue
// position of its segment's first entry (mul = 1 path queue, 2 shadow
// queue) and sets its first entry's offset in that segment and the
// segment's entry count.
template <class View>
__device__ __forceinline__ uint32_t unit_segment(const View& v, int ci, uint32_t uc, uint32_t mul, uint32_t& first,
                                                 uint32_t& lim) {
  uint32_t acc = 0;
  int x = 0;
  for (; x < kQSeg - 1; ++x) {
    const uint32_t n = (v.cnt[ci][x] + 63u) >> 6;
    if (uc < acc + n) break;
    acc += n;
  }
  first = (uc - acc) * 64u;
  lim = v.cnt[ci][x];
  const auto& ck = v.ch[ci];
  return mul * (static_cast<uint32_t>(ck.qbase) + static_cast<uint32_t>(x) * static_cast<uint32_t>(ck.qseg));
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }


}  // namespace xnh
