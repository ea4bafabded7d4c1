// dbsdf.h — principled BSDF on the device: diffuse, GGX conductor, GGX and
// delta dielectric, the diffuse-like subsurface lobe, NEE eval/pdf and lobe
// selection, with the semantics of material/bsdf.h:30-708.
//
// RNG draw order: the reference passes two draws straight into a call
// (bsdf.h:252, 347, 429, 566) and is built with g++, which evaluates those
// call arguments right to left, so the SECOND draw becomes u1. The kernels
// draw explicitly in that order.
//
// Transcendentals (cos, sin, pow) are the device's and may differ from
// glibc by an ulp; everything else rounds as the host does.
#pragma once
#include "../common/dev_types.h"
#include "dmath.h"
#include "xenon_hip.h"

namespace xnh {

// Material as six float4 in HBM (kMatVecs):
//   {base.rgb, metallic} {ior, alpha, alpha_x, alpha_y} {f0.rgb, subsurface}
//   {subsurface.rgb, flags} {ms_k1, ms_k2, ms_f.r, ms_f.g} {ms_f.b, 0, 0, 0}
// The last two hold the parts of the multiple-scattering compensation
// (bsdf.h:212-249) that depend on the material alone, computed at upload
// with the same float operations in the same order: ms_k1 = 5 exp(-2.69 a),
// ms_k2 = 1 + 22.7 a^1.5 and ms_f = favg^2 E_avg / max(1 - favg.r (1 - E_avg), 1e-4).
struct DMat {
  f3 base, f0, ss, ms_f;
  float metallic, ior, alpha, ax, ay, sss, ms_k1, ms_k2;
  uint32_t flags;
  __device__ __forceinline__ bool conductor() const { return flags & XNH_MAT_CONDUCTOR; }
  __device__ __forceinline__ bool transmissive() const { return flags & XNH_MAT_TRANSMISSIVE; }
  __device__ __forceinline__ bool has_sss() const { return flags & XNH_MAT_SUBSURFACE; }
  __device__ __forceinline__ bool delta() const { return flags & XNH_MAT_DELTA; }
};

__device__ __forceinline__ DMat load_mat(const float4* mats, int id) {
  const float4* r = mats + kMatVecs * id;
  const float4 a = r[0], b = r[1], c = r[2], d = r[3], e = r[4], g = r[5];
  DMat m;
  m.base = xyz(a);
  m.metallic = a.w;
  m.ior = b.x;
  m.alpha = b.y;
  m.ax = b.z;
  m.ay = b.w;
  m.f0 = xyz(c);
  m.sss = c.w;
  m.ss = xyz(d);
  m.flags = __float_as_uint(d.w);
  m.ms_k1 = e.x;
  m.ms_k2 = e.y;
  m.ms_f = f3{e.z, e.w, g.x};
  return m;
}

struct BSample {
  f3 wi, f;
  float pdf;
  bool delta;
};

__device__ __forceinline__ float c2t(f3 w) { return w.z * w.z; }
__device__ __forceinline__ float s2t(f3 w) { return smax(0.f, 1.f - c2t(w)); }
__device__ __forceinline__ float t2t(f3 w) {
  const float c2 = c2t(w);
  return (c2 < 1e-8f) ? 0.f : div_r(s2t(w), c2, recip(c2));
}
// cos and sin of the azimuth (their squares are what is used: a component too
// small for div_r adds nothing to them).
__device__ __forceinline__ void azimuth(f3 w, float& cp, float& sp) {
  const float s = sqrt_r(s2t(w)), r = recip(s);
  cp = (s == 0.f) ? 1.f : sclamp(div_r(w.x, s, r), -1.f, 1.f);
  sp = (s == 0.f) ? 0.f : sclamp(div_r(w.y, s, r), -1.f, 1.f);
}

__device__ __forceinline__ float mis_power2(float a, float b) {
  const float a2 = a * a, b2 = b * b, s = a2 + b2;
  return (s > 0.f) ? a2 / s : 0.f;
}

constexpr float kPiD = 3.14159265358979323846f;
constexpr float kInvPiD = 1.f / kPiD;

__device__ __forceinline__ float D_ggx(f3 h, float ax, float ay) {
  const float c2 = c2t(h);
  if (c2 <= 0.f) return 0.f;
  float cp, sp;
  azimuth(h, cp, sp);
  const float ex = div_r(cp, ax, recip(ax)), ey = div_r(sp, ay, recip(ay));
  const float tn = (ex * ex + ey * ey) * t2t(h);
  const float d = c2 * c2 * (1.f + tn);
  return 1.f / (kPiD * ax * ay * d * d);
}
__device__ __forceinline__ float Lambda_ggx(f3 w, float ax, float ay) {
  const float t2 = t2t(w);
  if (t2 == 0.f) return 0.f;
  float cp, sp;
  azimuth(w, cp, sp);
  const float a2 = (cp * ax) * (cp * ax) + (sp * ay) * (sp * ay);
  return (-1.f + sqrt_r(1.f + a2 * t2)) * 0.5f;
}
__device__ __forceinline__ float fresnel_d(float ci, float ior) {
  ci = sclamp(ci, -1.f, 1.f);
  float ei = 1.f, et = ior, eta = recip(ior);   // eta = ei / et
  if (ci < 0.f) {
    ei = ior;
    et = 1.f;
    eta = ior;
    ci = -ci;
  }
  const float s2i = 1.f - ci * ci;
  const float s2o = eta * eta * s2i;
  if (s2o >= 1.f) return 1.f;
  const float ct = sqrt_r(smax(0.f, 1.f - s2o));
  const float da = (et * ci) + (ei * ct), de = (ei * ci) + (et * ct);
  const float rpa = div_r((et * ci) - (ei * ct), da, recip(da));
  const float rpe = div_r((ei * ci) - (et * ct), de, recip(de));
  return (rpa * rpa + rpe * rpe) * 0.5f;
}
__device__ __forceinline__ f3 fresnel_s(float c, f3 f0) {
  const float m = sclamp(1.f - c, 0.f, 1.f);
  const float m2 = m * m;
  return f0 + (splat(1.f) - f0) * (m2 * m2 * m);
}

__device__ __forceinline__ f3 cosine_dir(float u1, float u2) {
  const float r = sqrt_r(u1);
  const float phi = 2.0f * kPiD * u2;
  const SinCos sc = sincos_r(phi);
  return f3{r * sc.c, r * sc.s, sqrt_r(smax(0.0f, 1.0f - u1))};
}

// Heitz 2018 visible-normal sampling (bsdf.h:164-190).
__device__ __forceinline__ f3 vndf(f3 wo, float ax, float ay, float u1, float u2) {
  const f3 vh = normalize(f3{ax * wo.x, ay * wo.y, wo.z});
  const float l2 = vh.x * vh.x + vh.y * vh.y;
  const f3 t1 = (l2 > 1e-7f) ? f3{-vh.y, vh.x, 0.f} * recip(sqrt_r(l2)) : f3{1.f, 0.f, 0.f};
  const f3 t2 = cross(vh, t1);
  const float r = sqrt_r(u1);
  const float phi = 2.0f * kPiD * u2;
  const SinCos sc = sincos_r(phi);
  const float p1 = r * sc.c;
  float p2 = r * sc.s;
  const float s = 0.5f * (1.0f + vh.z);
  p2 = (1.0f - s) * sqrt_r(smax(0.f, 1.0f - p1 * p1)) + s * p2;
  const f3 nh = p1 * t1 + p2 * t2 + sqrt_any(smax(0.f, 1.0f - p1 * p1 - p2 * p2)) * vh;
  return normalize(f3{ax * nh.x, ay * nh.y, smax(0.f, nh.z)});
}
// The pdf of h from its D and G1 (bsdf.h:192-199).
__device__ __forceinline__ float vndf_pdf(f3 wo, f3 h, float D, float g1) {
  const float co = fabsf(wo.z);
  if (co < 1e-8f) return 0.f;
  return D * g1 * smax(0.f, dot(wo, h)) / co;
}

// bsdf.h:212-249 per evaluation: the directional albedo E(c) and the
// compensation factor, with the material's constant parts precomputed.
__device__ __forceinline__ float ms_E(float c, const DMat& m, float rk2) {
  const float e = 1.0f - div_r(pow_r(1.0f - c, m.ms_k1), m.ms_k2, rk2);
  return sclamp(e, 0.f, 1.f);
}
__device__ __forceinline__ f3 ms_comp(const DMat& m, float co, float ci) {
  const float rk2 = recip(m.ms_k2);   // (k2 >= 1; a quotient too small for div_r is lost in 1 - e)
  const float eo = ms_E(fabsf(co), m, rk2), ei = ms_E(fabsf(ci), m, rk2);
  const float c = (1.f - eo) * (1.f - ei);
  const float b = smax(eo * ei, 1e-4f), r = recip(b);
  const f3 n = m.ms_f * c;
  return splat(1.f) + f3{div_r(n.x, b, r), div_r(n.y, b, r), div_r(n.z, b, r)};
}

// ---- lobes ------------------------------------------------------------------
__device__ __forceinline__ f3 diffuse_f(f3 wi, const DMat& m) {
  if (wi.z <= 0.f) return splat(0.f);
  return m.base * (1.f - m.metallic) * kInvPiD;
}
__device__ __forceinline__ float diffuse_pdf(f3 wi) { return (wi.z <= 0.f) ? 0.f : wi.z * kInvPiD; }

__device__ __forceinline__ f3 refl_F(float ch, const DMat& m) {
  if (m.conductor()) return fresnel_s(fabsf(ch), m.f0);
  return splat(fresnel_d(ch, m.ior));
}
// The value and the pdf of the reflection lobe. Both need the half vector, D
// and Lambda(wo), and every caller needs both. Shading is bound by its
// instructions (VALU busy 85 %); evaluated together, with one inlined copy for
// all material classes and with sqrt_r, recip and div_r for the library's
// expansions, k_shade takes 4.04 -> 3.42 ms (Cornell box 512x512 at 64 spp) and
// 1.77 -> 1.26 ms (primitive scene 801x449 at 33 spp).
__device__ __forceinline__ void refl_eval(f3 wo, f3 wi, const DMat& m, f3& f, float& pdf) {
  f = splat(0.f);
  pdf = 0.f;
  if (wo.z <= 0.f || wi.z <= 0.f) return;
  const f3 h = normalize(wo + wi);
  if (h.z <= 0.f) return;
  const float D = D_ggx(h, m.ax, m.ay);
  const float lo = 1.f + Lambda_ggx(wo, m.ax, m.ay);
  const float oh = dot(wo, h);
  pdf = vndf_pdf(wo, h, D, recip(lo)) * (1.f / (4.f * fabsf(oh)));
  const float den = 4.f * wo.z * wi.z;
  if (den < 1e-8f) return;
  const float G = recip(lo + Lambda_ggx(wi, m.ax, m.ay));
  const f3 F = refl_F(oh, m);
  f = F * D * G * recip(den);
  if (!m.transmissive()) f = f * ms_comp(m, wo.z, wi.z);
}
__device__ __forceinline__ void trans_eval(f3 wo, f3 wi, const DMat& m, f3& f, float& pdf) {
  f = splat(0.f);
  pdf = 0.f;
  if (wo.z == 0.f || wi.z == 0.f) return;
  if (wo.z * wi.z > 0.f) return;
  const float eta = (wo.z > 0.f) ? (1.f / m.ior) : m.ior;
  f3 h = normalize(wo + eta * wi);
  if (h.z < 0.f) h = -h;
  const float oh = dot(wo, h), ih = dot(wi, h);
  if (oh * ih >= 0.f) return;
  const float D = D_ggx(h, m.ax, m.ay);
  const float lo = 1.f + Lambda_ggx(wo, m.ax, m.ay);
  const float den = oh + eta * ih;
  const float den2 = den * den;
  if (fabsf(den) < 1e-8f) return;
  pdf = vndf_pdf(wo, h, D, recip(lo)) * fabsf((eta * eta * ih) / den2);
  const float co = fabsf(wo.z), ci = fabsf(wi.z);
  if (co < 1e-8f || ci < 1e-8f) return;
  const float G = recip(lo + Lambda_ggx(wi, m.ax, m.ay));
  const float F = fresnel_d(oh, m.ior);
  const float fac = fabsf(oh * ih) * (eta * eta) / (co * ci * den2);
  f = m.base * ((1.f - F) * D * G * fac);
}
__device__ __forceinline__ f3 sss_f(f3 wi, const DMat& m) {
  if (wi.z <= 0.f) return splat(0.f);
  return lerp3(m.base, m.ss, m.sss) * (1.f - m.metallic) * kInvPiD;
}

// True when the BSDF is exactly Lambertian: an opaque, non-metal dielectric
// with F0 = 0 (IOR 1), whose sampler always takes the cosine lobe
// (bsdf.h:666-708 with a zero specular weight) and whose NEE terms reduce to
// the diffuse lobe. Path guiding mixes its sampler with this one.
__device__ __forceinline__ bool lambert_exact(const DMat& m) {
  return (m.flags & (XNH_MAT_DELTA | XNH_MAT_CONDUCTOR | XNH_MAT_TRANSMISSIVE | XNH_MAT_SUBSURFACE)) == 0u &&
         m.f0.x == 0.f;
}

// True when the reflection lobe of a dielectric has weight 0 (f0.x = 0, IOR 1)
// and both its value and its pdf are finite for this pair, so that it adds
// nothing. h.z >= (wo.z + wi.z) / 2 >= 2^-6 and ax ay >= 2^-20 bound D by
// 2^66 and 1 / (4 wo.h) by 16; the evaluations divide by no less than 1e-8;
// cosines of at most 1 and an alpha and compensation that are not extreme
// keep the compensation below 2^37. Outside these bounds (and for NaN) the lobe
// is evaluated. Cornell box 512x512 at 64 spp: k_shade 3.42 -> 3.18 ms.
__device__ __forceinline__ bool refl_adds_nothing(f3 wo, f3 wi, const DMat& m) {
  return m.f0.x == 0.f && wo.z <= 1.f && wi.z <= 1.f && wo.z + wi.z >= 0x1p-5f && m.ax * m.ay >= 0x1p-20f &&
         m.alpha >= 0.f && m.alpha <= 16.f && m.ior == 1.f &&
         smax(smax(fabsf(m.ms_f.x), fabsf(m.ms_f.y)), fabsf(m.ms_f.z)) <= 0x1p20f;
}

// NEE: the value and the pdf summed over the non-delta lobes
// (bsdf.h:601-657), for a non-delta material and wi above the surface (where
// the transmission lobe has no part).
__device__ __forceinline__ void nee_eval(f3 wo, f3 wi, const DMat& m, f3& f, float& pdf) {
  if (m.has_sss() && !m.conductor() && !m.transmissive()) {
    f = sss_f(wi, m);
    pdf = diffuse_pdf(wi);
    return;
  }
  const bool opaque = !m.conductor() && !m.transmissive();
  f = splat(0.f);
  pdf = 0.f;
  if (!(opaque && refl_adds_nothing(wo, wi, m))) refl_eval(wo, wi, m, f, pdf);
  if (m.conductor()) return;
  if (m.transmissive()) {
    pdf = fresnel_d(fabsf(wo.z), m.ior) * pdf;
    return;
  }
  const float ws = m.f0.x, wd = 1.f - ws;
  f = diffuse_f(wi, m) * wd + f * ws;
  pdf = diffuse_pdf(wi) * wd + pdf * ws;
}

__device__ __forceinline__ bool sample_diffuse_like(f3 wo, f3 color, const DMat& m, Rng& rng, BSample& s) {
  const float first = rng.f();
  const float second = rng.f();
  s.wi = cosine_dir(second, first);
  if (wo.z < 0.f) s.wi.z = -s.wi.z;
  s.pdf = fabsf(s.wi.z) * kInvPiD;
  if (s.pdf < 1e-8f) return false;
  s.f = color * (1.f - m.metallic) * kInvPiD;
  s.delta = false;
  return true;
}
__device__ __forceinline__ bool sample_refl(f3 wo, const DMat& m, Rng& rng, BSample& s) {
  if (wo.z <= 0.f) return false;
  const float first = rng.f();
  const float second = rng.f();
  const f3 h = vndf(wo, m.ax, m.ay, second, first);
  if (h.z <= 0.f) return false;
  s.wi = reflect(-wo, h);
  if (s.wi.z <= 0.f) return false;
  refl_eval(wo, s.wi, m, s.f, s.pdf);
  s.delta = false;
  return !(s.pdf < 1e-8f);
}
__device__ __forceinline__ bool sample_trans(f3 wo, const DMat& m, Rng& rng, BSample& s) {
  if (fabsf(wo.z) < 1e-8f) return false;
  const float first = rng.f();
  const float second = rng.f();
  f3 h = vndf(wo, m.ax, m.ay, second, first);
  if (h.z < 0.f) h = -h;
  const float eta = (wo.z > 0.f) ? (1.f / m.ior) : m.ior;
  const float oh = dot(wo, h);
  const float s2o = smax(0.f, 1.f - oh * oh);
  const float s2i = eta * eta * s2o;
  if (s2i >= 1.f) return false;
  const float ci = sqrt_r(smax(0.f, 1.f - s2i));
  const float sg = (oh > 0.f) ? 1.f : -1.f;
  s.wi = normalize((-eta * wo) + (eta * oh - sg * ci) * h);
  if (wo.z * s.wi.z > 0.f) return false;
  trans_eval(wo, s.wi, m, s.f, s.pdf);
  s.delta = false;
  return !(s.pdf < 1e-8f);
}
__device__ __forceinline__ bool sample_mirror(f3 wo, const DMat& m, BSample& s) {
  if (fabsf(wo.z) < 1e-8f) return false;
  const f3 n{0.f, 0.f, (wo.z > 0.f) ? 1.f : -1.f};
  s.wi = reflect(-wo, n);
  const f3 F = m.conductor() ? fresnel_s(fabsf(wo.z), m.f0) : splat(fresnel_d(fabsf(wo.z), m.ior));
  const float ci = fabsf(s.wi.z);
  if (ci < 1e-8f) return false;
  s.f = F / ci;
  s.pdf = 1.f;
  s.delta = true;
  return true;
}
__device__ __forceinline__ bool sample_glass(f3 wo, const DMat& m, BSample& s) {
  if (fabsf(wo.z) < 1e-8f) return false;
  const float eta = (wo.z > 0.f) ? (1.f / m.ior) : m.ior;
  const f3 n{0.f, 0.f, (wo.z > 0.f) ? 1.f : -1.f};
  // Snell refraction of v = -wo about n (math/vec3.h:61-68)
  const f3 v = -wo;
  const float ci0 = -dot(normalize(v), n);
  const float s2 = eta * eta * (1.f - ci0 * ci0);
  if (s2 >= 1.f) return false;
  s.wi = normalize(eta * v + (eta * ci0 - sqrt_r(1.f - s2)) * n);
  const float F = fresnel_d(fabsf(wo.z), m.ior);
  const float ci = fabsf(s.wi.z);
  if (ci < 1e-8f) return false;
  s.f = m.base * ((1.f - F) * eta * eta / ci);
  s.pdf = 1.f;
  s.delta = true;
  return true;
}

// Lobe selection (bsdf.h:666-708).
__device__ __forceinline__ bool sample_bsdf(f3 wo, const DMat& m, Rng& rng, BSample& s) {
  if (m.delta()) {
    if (m.transmissive()) {
      const float F = fresnel_d(wo.z, m.ior);
      if (rng.f() < F) return sample_mirror(wo, m, s);
      return sample_glass(wo, m, s);
    }
    return sample_mirror(wo, m, s);
  }
  // one call of each sampler for all classes
  bool refl = m.conductor();
  float share = 1.f;   // the lobe's probability
  f3 color = m.base;
  if (!refl) {
    if (m.has_sss()) {
      color = lerp3(m.base, m.ss, m.sss);
    } else {
      const float ws = m.transmissive() ? fresnel_d(fabsf(wo.z), m.ior) : sclamp(m.f0.x, 0.f, 1.f);
      refl = rng.f() < ws;
      share = refl ? ws : 1.f - ws;
    }
  }
  bool ok;
  if (refl) ok = sample_refl(wo, m, rng, s);
  else if (m.transmissive() && !m.has_sss()) ok = sample_trans(wo, m, rng, s);
  else ok = sample_diffuse_like(wo, color, m, rng, s);
  s.pdf *= share;
  return ok;
}

}  // namespace xnh
