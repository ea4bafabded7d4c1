// dmath.h — device scalar math for the wavefront kernels.
//
// All HIP sources are compiled with -ffp-contract=off and the default
// correctly rounded fp32 division and square root, so +, -, *, /, sqrt
// round exactly as the reference's host code does (math/vec3.h:12-84,
// math/ray.h:95-113). Operators keep the reference's left-to-right
// association; that, not style, fixes their order.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace xnh {

struct f3 {
  float x, y, z;
};

// Loads through pointers known to address device (global) memory. Pointers
// read from memory (scene tables in the job list) are otherwise generic, and
// generic loads count against the LDS wait counter as well, so every LDS
// stack access would also wait for outstanding node fetches.
typedef float xv4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 gld4(const float4* p, size_t i) {
  const xv4 v = ((const __attribute__((address_space(1))) xv4*)p)[i];
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t gld1(const uint32_t* p, size_t i) {
  return ((const __attribute__((address_space(1))) uint32_t*)p)[i];
}
__device__ __forceinline__ void gst1(uint32_t* p, size_t i, uint32_t v) {
  ((__attribute__((address_space(1))) uint32_t*)p)[i] = v;
}

// Float cos, sin and pow evaluated in double and rounded once to
// float: the correctly rounded result except in rare double-rounding cases.
// The reference calls glibc's float functions (std::cos(float) etc. in
// material/bsdf.h and scene/environment.h), which compute in double
// internally and return the correctly rounded value for nearly every input;
// the device library's float versions differ from it in the last bit far
// more often, and a last-bit difference in a sampled direction can send a
// path elsewhere.
//
// The series are written out here: the device library's double functions
// serve every argument (long reductions, extended precision, a call each),
// and shading is bound by its instruction stream. Cornell box 512x512 at 64
// spp 12.18 -> 11.41 ms, mesh 1920x1080 at 256 spp 238.9 -> 231.7 ms,
// primitive scene 801x449 at 33 spp 6.39 -> 6.05 ms.

// cos and sin of x, |x| <= 8: x less the nearest multiple of pi / 2 (in two
// parts), Taylor polynomials to r^15 and r^16 (truncated below 1e-16 of the
// value for |r| <= pi / 4). Equal to the library's double functions rounded to
// float for all 2^24 arguments that the samplers form (2 pi k / 2^24).
struct SinCos {
  float s, c;
};
__device__ __attribute__((noinline)) SinCos sincos_r(float xf) {
  const double x = xf, k = __builtin_rint(x * 0.63661977236758134308);
  const double r = __builtin_fma(-k, 6.12323399573676603587e-17, __builtin_fma(-k, 1.57079632679489655800, x));
  const double z = r * r;
  double a = -1.0 / 1307674368000.0;
  a = __builtin_fma(a, z, 1.0 / 6227020800.0);
  a = __builtin_fma(a, z, -1.0 / 39916800.0);
  a = __builtin_fma(a, z, 1.0 / 362880.0);
  a = __builtin_fma(a, z, -1.0 / 5040.0);
  a = __builtin_fma(a, z, 1.0 / 120.0);
  a = __builtin_fma(a, z, -1.0 / 6.0);
  const float sr = static_cast<float>(__builtin_fma(a * z, r, r));
  double b = 1.0 / 20922789888000.0;
  b = __builtin_fma(b, z, -1.0 / 87178291200.0);
  b = __builtin_fma(b, z, 1.0 / 479001600.0);
  b = __builtin_fma(b, z, -1.0 / 3628800.0);
  b = __builtin_fma(b, z, 1.0 / 40320.0);
  b = __builtin_fma(b, z, -1.0 / 720.0);
  b = __builtin_fma(b, z, 1.0 / 24.0);
  b = __builtin_fma(b, z, -0.5);
  const float cr = static_cast<float>(__builtin_fma(b, z, 1.0));
  const int q = static_cast<int>(k);
  const float u = (q & 1) ? cr : sr, v = (q & 1) ? sr : cr;
  return SinCos{(q & 2) ? -u : u, ((q + 1) & 2) ? -v : v};
}

// x^y for a normal 0 < x <= 1 and 2^-10 <= y <= 2^10: 2^(y log2 x), with
// log2 m = 2 / ln 2 atanh((m - 1) / (m + 1)) for the mantissa in [sqrt 1/2,
// sqrt 2) and the exponential's Taylor series on [-ln 2 / 2, ln 2 / 2]. Other
// arguments go to the library. Against the library's double pow rounded to
// float, over every x, y = 1/3, 0.4, 0.8, 1.7, 2.31, 5: 6 to 39 of 1.07e9
// results differ (double-rounding cases).
__device__ __forceinline__ float pow_lib(float x, float y) {
  return static_cast<float>(pow(static_cast<double>(x), static_cast<double>(y)));
}
__device__ __attribute__((noinline)) float pow_r(float x, float y) {
  if (!(x >= 0x1p-126f && x <= 1.f && y >= 0x1p-10f && y <= 0x1p10f)) return pow_lib(x, y);
  const uint32_t bits = __float_as_uint(x);
  int e = static_cast<int>(bits >> 23) - 127;
  float m = __uint_as_float((bits & 0x7fffffu) | 0x3f800000u);
  if (m > 1.41421356f) {
    m *= 0.5f;
    e += 1;
  }
  const double md = m, t = md + 1.0;
  double r = __builtin_amdgcn_rcpf(m + 1.f);
  r = __builtin_fma(__builtin_fma(-t, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-t, r, 1.0), r, r);
  const double s = (md - 1.0) * r, z = s * s;
  double p = 1.0 / 21.0;
  p = __builtin_fma(p, z, 1.0 / 19.0);
  p = __builtin_fma(p, z, 1.0 / 17.0);
  p = __builtin_fma(p, z, 1.0 / 15.0);
  p = __builtin_fma(p, z, 1.0 / 13.0);
  p = __builtin_fma(p, z, 1.0 / 11.0);
  p = __builtin_fma(p, z, 1.0 / 9.0);
  p = __builtin_fma(p, z, 1.0 / 7.0);
  p = __builtin_fma(p, z, 1.0 / 5.0);
  p = __builtin_fma(p, z, 1.0 / 3.0);
  const double l2 = __builtin_fma(__builtin_fma(p * z, s, s), 2.88539008177792681472, static_cast<double>(e));
  const double w = static_cast<double>(y) * l2, n = __builtin_rint(w), g = (w - n) * 0.693147180559945309417;
  double q = 1.0 / 6227020800.0;
  q = __builtin_fma(q, g, 1.0 / 479001600.0);
  q = __builtin_fma(q, g, 1.0 / 39916800.0);
  q = __builtin_fma(q, g, 1.0 / 3628800.0);
  q = __builtin_fma(q, g, 1.0 / 362880.0);
  q = __builtin_fma(q, g, 1.0 / 40320.0);
  q = __builtin_fma(q, g, 1.0 / 5040.0);
  q = __builtin_fma(q, g, 1.0 / 720.0);
  q = __builtin_fma(q, g, 1.0 / 120.0);
  q = __builtin_fma(q, g, 1.0 / 24.0);
  q = __builtin_fma(q, g, 1.0 / 6.0);
  q = __builtin_fma(q, g, 0.5);
  q = __builtin_fma(q, g, 1.0);
  q = __builtin_fma(q, g, 1.0);
  return static_cast<float>(__builtin_ldexp(q, static_cast<int>(n)));
}

// 1 / x, correctly rounded (the value of the division) in four instructions
// instead of ten: the hardware's approximation and one Newton step with fused
// multiply-adds (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990), and the division's own fix-up of zeros,
// infinities and NaN. Equal to the division on gfx950 for every float but
// those below 2^-126 and from 2^126 on, so it is for arguments that cannot lie
// there: square roots, and sums with a term of 1. The mesh scene
// above: 231.7 -> 228.3 ms.
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r), x, 1.f);
}

// a / b with r = recip(b): one correction of a * r (Markstein, as above). The
// value of the division where b, the quotient and their product are normal
// floats some way from the ends of the range; a zero quotient can lose its
// sign. One reciprocal serves several dividends.
__device__ __forceinline__ float div_r(float a, float b, float r) {
  const float q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}

// The value of sqrtf for zero, infinity and x >= 2^-96, in seven instructions
// instead of fifteen: x * rsq(x) and one Newton step. Compared with sqrtf on
// gfx950 for every such float.
__device__ __forceinline__ float sqrt_r(float x) {
  const float r = __builtin_amdgcn_rsqf(x), s = x * r;
  const float v = __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * r, s);
  return __builtin_amdgcn_classf(x, 0x260) ? x : v;   // -0, +0, +inf
}
// The value of sqrtf.
__device__ __forceinline__ float sqrt_any(float x) {
  float v = sqrt_r(x);
  if (x > 0.f && x < 0x1p-96f) {
    asm volatile("");   // (keeps the library's expansion out of the common path)
    v = sqrtf(x);
  }
  return v;
}

__device__ __forceinline__ f3 mk(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ f3 splat(float s) { return f3{s, s, s}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return f3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return f3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator*(f3 a, f3 b) { return f3{a.x * b.x, a.y * b.y, a.z * b.z}; }
__device__ __forceinline__ f3 operator/(f3 a, f3 b) { return f3{a.x / b.x, a.y / b.y, a.z / b.z}; }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return f3{a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return f3{a.x * s, a.y * s, a.z * s}; }
// Division by a scalar multiplies by its reciprocal (math/vec3.h:29).
__device__ __forceinline__ f3 operator/(f3 a, float s) {
  const float r = 1.f / s;
  return f3{a.x * r, a.y * r, a.z * r};
}
__device__ __forceinline__ f3 operator-(f3 a) { return f3{-a.x, -a.y, -a.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
  return f3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float len2(f3 a) { return a.x * a.x + a.y * a.y + a.z * a.z; }
__device__ __forceinline__ f3 normalize(f3 a) { return a * recip(sqrt_any(len2(a))); }
__device__ __forceinline__ f3 lerp3(f3 a, f3 b, float t) { return a + t * (b - a); }
__device__ __forceinline__ f3 reflect(f3 v, f3 n) { return v - 2.f * dot(v, n) * n; }
__device__ __forceinline__ float comp(f3 v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }

// std::max / std::min / std::clamp value semantics (first operand kept on
// ties and NaN comparisons), used wherever the reference calls them.
__device__ __forceinline__ float smax(float a, float b) { return (a < b) ? b : a; }
__device__ __forceinline__ float smin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float sclamp(float v, float lo, float hi) { return (v < lo) ? lo : ((hi < v) ? hi : v); }
// SSE MINPS / MAXPS lane semantics (geometry/blas.cpp:40-70).
__device__ __forceinline__ float xmin(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float xmax(float a, float b) { return a > b ? a : b; }

__device__ __forceinline__ bool finite3(f3 v) { return isfinite(v.x) && isfinite(v.y) && isfinite(v.z); }

// PCG32 XSH-RR (camera/sampler.h:13-36), stream increment 1.
struct Rng {
  uint64_t s;
  __device__ __forceinline__ uint32_t u32() {
    const uint64_t old = s;
    s = old * 6364136223846793005ULL + 1ULL;
    const uint32_t xs = static_cast<uint32_t>(((old >> 18u) ^ old) >> 27u);
    const uint32_t rot = static_cast<uint32_t>(old >> 59u);
    return (xs >> rot) | (xs << ((~rot + 1u) & 31u));
  }
  __device__ __forceinline__ float f() { return static_cast<float>(u32() >> 8) * (1.f / 16777216.f); }
};

// seed_pcg(seed, 0): state 0, one step, add the seed, one step.
__device__ __forceinline__ Rng rng_for(uint64_t seed) {
  Rng r{0};
  r.u32();
  r.s += seed;
  r.u32();
  return r;
}

// Duff et al. 2017 frame (math/ray.h:95-113).
struct Frame {
  f3 t, b, n;
  __device__ __forceinline__ explicit Frame(f3 nn) : n(nn) {
    const float s = (n.z >= 0.f) ? 1.f : -1.f;
    const float a = -recip(s + n.z);
    const float c = n.x * n.y * a;
    t = f3{1.f + s * n.x * n.x * a, s * c, -s * n.x};
    b = f3{c, s + n.y * n.y * a, -n.y};
  }
  __device__ __forceinline__ f3 world(f3 l) const { return l.x * t + l.y * b + l.z * n; }
  __device__ __forceinline__ f3 local(f3 w) const { return f3{dot(w, t), dot(w, b), dot(w, n)}; }
};

// Offset along the geometric normal toward `dir` (math/ray.h:22-26).
__device__ __forceinline__ f3 offset_origin(f3 p, f3 ng, f3 dir, float eps) {
  f3 n = ng;
  if (dot(n, dir) < 0.f) n = -n;
  return p + n * eps;
}

__device__ __forceinline__ f3 xyz(float4 v) { return f3{v.x, v.y, v.z}; }

}  // namespace xnh
