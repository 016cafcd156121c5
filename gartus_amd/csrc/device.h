// device.h — device-side math, RNG, BSDFs, light and environment sampling
// for the wavefront path tracer (gfx950, FP32).
//
// Arithmetic follows the reference (cited per function) in FP32. Constants
// that the reference compares against f64::EPSILON keep that value.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"

namespace gtd {

constexpr float EPS = 2.220446049250313e-16f;  // f64::EPSILON as a float
constexpr float PI = 3.14159265358979323846f;
constexpr float TAU = 6.28318530717958647692f;
constexpr float INF = __builtin_huge_valf();
constexpr float SHADOW_ACNE = 0.001f;          // raytracing.rs:146, object.rs:1163

struct f3 {
  float x, y, z;
};
__device__ __forceinline__ f3 mk(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator-(f3 a) { return {-a.x, -a.y, -a.z}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
// Correctly rounded FP32 reciprocals, quotients and square roots for operands
// whose results and remainders stay in the normal range, as those of a traced
// ray do: the compiler's general forms also scale their operands and handle
// zeros, infinities and denormals, and cannot share one divisor's reciprocal.
// The refinement steps are Markstein's (IBM J. Res. Dev. 34, 1990): with fma, a
// residual is exact, so a quotient or root within an ulp of the true value comes
// out correctly rounded. The tests compare reciprocals and roots with the
// operators over every operand of the ranges stated here, quotients over every
// divisor with sampled numerators: the same bits, but that a zero quotient is
// always +0 and an infinite numerator gives NaN. Vector instructions: 7 for a
// reciprocal, 5 for each further quotient of the same divisor and 8 for a root,
// against about 10, 10 and 14. Together with straight-line primitive tests, a sky
// lookup without fmod and table cosines, on one MI355X: 720p terrain 13.7 ->
// 13.1 ms, 12 small scenes 5.3 -> 5.0 ms, 1080p GGX/environment 13.1 -> 12.8 ms.
__device__ __forceinline__ float rcp_rn(float d) {  // 2^-96 <= |d| < 2^126
  float r = __builtin_amdgcn_rcpf(d);
  r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
  const float q = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
  return __builtin_fmaf(__builtin_fmaf(-d, q, 1.0f), r, q);
}
// 1 / d for |d| >= 2^-96. The reciprocal of 2^126 and more is subnormal, which rcp_rn cannot make: then the whole
// wave divides. No ray of an ordinary scene gets there: one comparison and a branch not taken, kept out of line by the
// empty asm (as a choice between the two, 12 small scenes took 4.93 ms for 4.90).
__device__ __forceinline__ bool beyond_rcp(float d) { return __ballot(!(fabsf(d) < 0x1p126f)) != 0ull; }
__device__ __forceinline__ float reciprocal(float d) {
  float r = rcp_rn(d);
  if (__builtin_expect(beyond_rcp(d), 0)) {
    asm volatile("" ::: "memory");
    r = 1.0f / d;
  }
  return r;
}
// n / d, with rd = reciprocal(d) (from |d| = 2^126 on rd has fewer bits and the quotient may be an ulp off).
__device__ __forceinline__ float div_rn(float n, float d, float rd) {
  float q = n * rd;
  q = __builtin_fmaf(__builtin_fmaf(-d, q, n), rd, q);
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), rd, q);
}
__device__ __forceinline__ float sqrt_rn(float x) {
  if (!(x >= 0x1p-96f && x < 0x1p126f)) return sqrtf(x);
  const float y = __builtin_amdgcn_rsqf(x);
  float s = x * y, h = 0.5f * y;
  const float e = __builtin_fmaf(-h, s, 0.5f);
  h = __builtin_fmaf(h, e, h);
  s = __builtin_fmaf(s, e, s);
  return __builtin_fmaf(__builtin_fmaf(-s, s, x), h, s);
}
__device__ __forceinline__ f3 operator/(f3 a, float s) { return {a.x / s, a.y / s, a.z / s}; }
constexpr float INV_PI = 1.0f / PI, INV_TAU = 1.0f / TAU;  // reciprocals for div_rn

// n / d and n % d for n < 2^31 by a multiplication: mul = floor(2^shift / d) + 1 with
// shift = 31 + ceil(log2 d) (Granlund and Montgomery, PLDI 1994).
struct Div31 {
  uint32_t d, mul, shift;
};
// Div31 of d in [1, 2^31].
inline Div31 make_div31(uint32_t d) {
  uint32_t l = 0;
  while ((uint64_t(1) << l) < d) ++l;
  return {d, uint32_t((uint64_t(1) << (31 + l)) / d + 1), 31 + l};
}
__device__ __forceinline__ uint32_t div31(uint32_t n, const Div31& k, uint32_t* rem) {
  const uint32_t q = uint32_t((uint64_t(n) * k.mul) >> k.shift);
  *rem = n - q * k.d;
  return q;
}
__device__ __forceinline__ f3 mul(f3 a, f3 b) { return {a.x * b.x, a.y * b.y, a.z * b.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float len2(f3 a) { return dot(a, a); }
__device__ __forceinline__ f3 normalized(f3 a) {  // vector.rs:151-158
  float l = sqrt_rn(len2(a));
  if (l < EPS) return {0.f, 0.f, 0.f};
  if (!(l < 0x1p126f)) return a / l;
  // no component is larger than l, so only the sign of a zero is left to restore (div_rn makes +0 of -0); plain
  // quotients here took the Cornell frame from 3.70 to 3.74 ms
  const float r = rcp_rn(l);
  return {copysignf(div_rn(a.x, l, r), a.x), copysignf(div_rn(a.y, l, r), a.y), copysignf(div_rn(a.z, l, r), a.z)};
}
__device__ __forceinline__ f3 reflected(f3 d, f3 n) { return d - 2.0f * dot(d, n) * n; }  // vector.rs:162
__device__ __forceinline__ f3 refracted(f3 d, f3 n, float eta) {  // vector.rs:168-173
  float c = fminf(dot(-d, n), 1.0f);
  f3 perp = eta * (d + c * n);
  f3 par = -sqrt_rn(fabsf(1.0f - len2(perp))) * n;
  return perp + par;
}
__device__ __forceinline__ bool finite3(f3 a) { return isfinite(a.x) && isfinite(a.y) && isfinite(a.z); }
__device__ __forceinline__ float clampf(float x, float lo, float hi) { return x < lo ? lo : (x > hi ? hi : x); }
__device__ __forceinline__ float pow5(float x) { float x2 = x * x; float x4 = x2 * x2; return x * x4; }
__device__ __forceinline__ f3 ld3(const float* p) { return {p[0], p[1], p[2]}; }
// A table in device memory that no kernel writes, at a wave-uniform address,
// as constant memory: its fields load as scalars, and the compiler takes the
// pointers among them for global ones. (Through generic pointers it would use
// flat instructions, which also occupy the LDS path and its wait counter.)
template <class T>
__device__ __forceinline__ const T& as_constant(const T* p) {
  typedef const __attribute__((address_space(4))) T* P;
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(a)), hi = __builtin_amdgcn_readfirstlane(uint32_t(a >> 32));
  return *(const T*)(P)(uint64_t(hi) << 32 | lo);
}

// ---- RNG: SplitMix64 (random.rs:23-29) -------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}
__device__ __forceinline__ uint64_t pixel_seed(uint64_t seed, uint32_t x, uint32_t y) {  // camera.rs:1720-1727
  return mix64(seed ^ (uint64_t(x) * 0x9E3779B97F4A7C15ULL) ^ (uint64_t(y) * 0xD1B54A32D192ED03ULL));
}
// Per-(pixel, sample, dimension) stream key; dimension 0 = camera, 1+b = bounce b.
__device__ __forceinline__ uint64_t stream_seed(uint64_t key, uint32_t sample, uint32_t dim) {
  return mix64(key ^ (uint64_t(sample + 1) * 0xD6E8FEB86659FD93ULL) ^ (uint64_t(dim + 1) * 0xA0761D6478BD642FULL));
}
struct Rng {
  uint64_t s;
  // random_double (random.rs:56-59) at float precision: the top 24 bits.
  __device__ __forceinline__ float next() {
    s += 0x9e3779b97f4a7c15ULL;
    return float(uint32_t(mix64(s) >> 40)) * 5.9604644775390625e-8f;
  }
  __device__ __forceinline__ uint64_t next_u64() {  // next_u64 (random.rs:23-29)
    s += 0x9e3779b97f4a7c15ULL;
    return mix64(s);
  }
  __device__ __forceinline__ float range(float lo, float hi) { return lo + (hi - lo) * next(); }
  __device__ __forceinline__ f3 unit_vector_spherical() {  // random.rs:107-115
    float r1 = next(), r2 = next();
    float z = 1.0f - 2.0f * r2;
    float radius = sqrt_rn(1.0f - z * z);
    float phi = TAU * r1;
    float s, c;
    sincosf(phi, &s, &c);
    return {c * radius, s * radius, z};
  }
  __device__ __forceinline__ f3 cosine_direction() {  // random.rs:119-126
    float r1 = next(), r2 = next();
    float phi = TAU * r1;
    float radius = sqrt_rn(r2);
    float s, c;
    sincosf(phi, &s, &c);
    return {c * radius, s * radius, sqrt_rn(1.0f - r2)};
  }
  __device__ __forceinline__ f3 in_unit_disk() {  // random.rs:141-152
    for (;;) {
      float a = range(-1.0f, 1.0f);
      float b = range(-1.0f, 1.0f);
      if (a * a + b * b < 1.0f) return {a, b, 0.0f};
    }
  }
};

// ---- orthonormal basis and PDFs (geometry.rs:122-137, sampling.rs) ----------
struct Onb {
  f3 u, v, w;
  __device__ __forceinline__ f3 local(f3 l) const { return l.x * u + l.y * v + l.z * w; }
};
__device__ __forceinline__ bool onb_from_w(f3 axis, Onb* o) {
  f3 w = normalized(axis);
  if (len2(w) <= EPS) return false;
  f3 a = fabsf(w.x) > 0.9f ? mk(0.f, 1.f, 0.f) : mk(1.f, 0.f, 0.f);
  f3 v = normalized(cross(w, a));
  o->u = cross(w, v);
  o->v = v;
  o->w = w;
  return true;
}
__device__ __forceinline__ float ggx_alpha(float r) {  // sampling.rs:310-312
  float c = clampf(r, 0.f, 1.f);
  return fmaxf(c * c, 1.0e-4f);
}
// sampling.rs:229-241. The reference's denominator cos^2 (a^2 - 1) + 1 is
// evaluated as sin^2 + a^2 cos^2 with sin^2 = |n x h|^2 from the vectors:
// the same value for unit n and h, but free of the cancellation that makes
// the FP32 form useless near the peak of a smooth lobe (at roughness 0.02,
// a^2 = 1.6e-7 is a couple of ulps of 1).
__device__ __forceinline__ float ggx_D(float ndh, float sin2, float roughness) {
  if (!isfinite(ndh) || ndh <= 0.f) return 0.f;
  float alpha = ggx_alpha(roughness);
  float a2 = alpha * alpha;
  float den = sin2 + a2 * (ndh * ndh);
  if (den <= EPS) return 0.f;
  return a2 / (PI * den * den);
}
__device__ __forceinline__ float smith_g1(float ndd, float roughness) {  // sampling.rs:314-322
  if (!isfinite(ndd) || ndd <= 0.f) return 0.f;
  float alpha = ggx_alpha(roughness);
  float a2 = alpha * alpha;
  return 2.0f * ndd / (ndd + sqrt_rn(a2 + (1.0f - a2) * ndd * ndd));
}
__device__ __forceinline__ float schlick(float c, float f0) {  // sampling.rs:255-261
  f0 = clampf(f0, 0.f, 1.f);
  return f0 + (1.0f - f0) * pow5(1.0f - clampf(c, 0.f, 1.f));
}
// HenyeyGreensteinPdf::phase_value (sampling.rs:126-136)
__device__ __forceinline__ float hg_phase(float cosine, float g) {
  if (!isfinite(cosine) || !isfinite(g) || fabsf(g) >= 1.0f) return 0.f;
  const float den = 1.0f + g * g - 2.0f * g * clampf(cosine, -1.f, 1.f);
  if (den <= EPS) return 0.f;
  return (1.0f - g * g) / (4.0f * PI * (den * sqrt_rn(den)));
}
// The material pdfs (MaterialPdf, pdf.rs:46-104): CosinePdf (sampling.rs:48-84),
// GgxReflectionPdf (:174-308), SpherePdf (:31-41), HenyeyGreensteinPdf (:91-166).
enum { PDF_COSINE = 0, PDF_GGX = 1, PDF_SPHERE = 2, PDF_HG = 3 };
struct MatPdf {
  Onb basis;
  f3 outgoing;
  float roughness, alpha;
  float g;
  uint32_t kind;
  __device__ float value(f3 d) const {
    if (kind == PDF_SPHERE) return 1.0f / (4.0f * PI);
    if (kind == PDF_HG) {
      const float l = sqrt_rn(len2(d));
      if (l <= EPS) return 0.f;
      return hg_phase(dot(d, basis.w) / l, g);
    }
    if (kind == PDF_COSINE) {
      float l = sqrt_rn(len2(d));
      if (l <= EPS) return 0.f;
      float c = dot(d, basis.w) / l;
      return c <= 0.f ? 0.f : div_rn(c, PI, INV_PI);
    }
    f3 in = normalized(d);
    if (len2(in) <= EPS || dot(in, basis.w) <= 0.f) return 0.f;
    f3 half = normalized(in + outgoing);
    float odh = dot(outgoing, half);
    if (len2(half) <= EPS || odh <= EPS) return 0.f;
    float ndh = dot(half, basis.w);
    return ggx_D(ndh, len2(cross(basis.w, half)), roughness) * fmaxf(ndh, 0.f) / (4.0f * fabsf(odh));
  }
  // *below (when given) reports a GGX reflection below the surface, where
  // the reference falls back to the outgoing direction.
  __device__ f3 generate(Rng& rng, bool* below = nullptr) const {
    if (kind == PDF_SPHERE) return rng.unit_vector_spherical();
    if (kind == PDF_HG) {  // sampling.rs:149-165
      const float r1 = rng.next(), r2 = rng.next();
      float ct;
      if (fabsf(g) < 1e-3f) {
        ct = 1.0f - 2.0f * r1;
      } else {
        const float term = (1.0f - g * g) / (1.0f - g + 2.0f * g * r1);
        ct = clampf((1.0f + g * g - term * term) / (2.0f * g), -1.f, 1.f);
      }
      const float st = sqrt_rn(fmaxf(1.0f - ct * ct, 0.f));
      float sn, cs;
      sincosf(2.0f * PI * r2, &sn, &cs);
      return basis.local(mk(cs * st, sn * st, ct));
    }
    if (kind == PDF_COSINE) return basis.local(rng.cosine_direction());
    float r1 = rng.next(), r2 = rng.next();
    float phi = 2.0f * PI * r1;
    float a2 = alpha * alpha;
    float cr2 = fminf(r2, 0.99999994f);
    float tan2 = a2 * cr2 / (1.0f - cr2);
    float ct = 1.0f / sqrt_rn(1.0f + tan2);
    // sin from tan: the reference's sqrt(1 - cos^2) cancels in FP32 when
    // tan^2 is a few ulps of 1, which would quantise a smooth lobe's angles
    float st = sqrt_rn(tan2) * ct;
    float s, c;
    sincosf(phi, &s, &c);
    f3 half = basis.local(mk(c * st, s * st, ct));
    f3 refl = reflected(-outgoing, normalized(half));
    const bool up = dot(refl, basis.w) > 0.f;
    if (below) *below = !up;
    return up ? refl : outgoing;
  }
};
// ggx_reflection_scattering_weight (material.rs:1686-1722)
__device__ __forceinline__ float ggx_weight(f3 n, f3 o, f3 i, float roughness, float f0) {
  n = normalized(n); o = normalized(o); i = normalized(i);
  float ndi = dot(n, i), ndo = dot(n, o);
  if (ndi <= 0.f || ndo <= 0.f) return 0.f;
  f3 half = normalized(i + o);
  if (len2(half) <= EPS) return 0.f;
  float ndh = dot(n, half), odh = dot(o, half);
  if (ndh <= 0.f || odh <= 0.f) return 0.f;
  float D = ggx_D(ndh, len2(cross(n, half)), roughness);
  float G = smith_g1(ndi, roughness) * smith_g1(ndo, roughness);
  f0 = clampf(f0, 0.f, 1.f);
  if (f0 <= EPS) return 0.f;
  float F = schlick(odh, f0) / f0;
  return D * G * F / (4.0f * ndo);
}

// ---- primitive intersection (geometry.rs, object.rs) -------------------------
struct PrimHit {
  float t, u, v;
};
__device__ __forceinline__ uint32_t meta_of(const float4& p0) { return __float_as_uint(p0.w); }

// hit_sphere_in_interval (object.rs:986-1013). The discriminant uses the
// perpendicular-distance form a*(r^2 - |oc - (h/a) d|^2), algebraically equal
// to h^2 - a*c and free of its cancellation in FP32.
__device__ __forceinline__ bool sphere_hit(f3 c, float r, f3 o, f3 d, float tmin, float tmax, float* root) {
  f3 oc = c - o;
  float a = len2(d);
  if (a <= EPS) return false;
  float h = dot(d, oc);
  f3 perp = oc - (h / a) * d;
  float disc = a * (r * r - len2(perp));
  if (disc < 0.f) return false;
  float sq = sqrt_rn(disc);
  float first = (h - sq) / a;
  if (tmin < first && first < tmax) { *root = first; return true; }
  float second = (h + sq) / a;
  if (tmin < second && second < tmax) { *root = second; return true; }
  return false;
}
// TriangleGeometry::hit_ray (geometry.rs:239-265)
__device__ __forceinline__ bool tri_hit(f3 v0, f3 e1, f3 e2, f3 o, f3 d, float tmin, float tmax, PrimHit* h) {
  f3 pvec = cross(d, e2);
  float det = dot(e1, pvec);
  if (fabsf(det) < 1e-10f) return false;
  float inv = reciprocal(det);
  f3 tvec = o - v0;
  float u = dot(tvec, pvec) * inv;
  if (!(u >= 0.f && u <= 1.f)) return false;
  f3 qvec = cross(tvec, e1);
  float v = dot(d, qvec) * inv;
  if (v < 0.f || u + v > 1.f) return false;
  float t = dot(e2, qvec) * inv;
  if (!(tmin < t && t < tmax)) return false;
  h->t = t; h->u = u; h->v = v;
  return true;
}
// QuadGeometry::hit_ray (geometry.rs:394-415); w = normal / |u x v|.
__device__ __forceinline__ bool quad_hit(f3 corner, f3 u, f3 v, f3 n, float inv_len, float nls, float plane_d,
                                         f3 o, f3 d, float tmin, float tmax, PrimHit* h) {
  if (nls <= EPS) return false;
  float denom = dot(n, d);
  if (fabsf(denom) < 1e-8f) return false;
  float t = (plane_d - dot(n, o)) / denom;
  if (!(tmin < t && t < tmax)) return false;
  f3 pp = (o + t * d) - corner;
  f3 w = n * inv_len;
  float a = dot(w, cross(pp, v));
  float b = dot(w, cross(u, pp));
  if (!(a >= 0.f && a <= 1.f) || !(b >= 0.f && b <= 1.f)) return false;
  h->t = t; h->u = a; h->v = b;
  return true;
}
// One primitive record against a ray interval; returns the root only.
__device__ __forceinline__ bool prim_test(const GPrim* __restrict__ prims, uint32_t k, f3 o, f3 d, float time,
                                          float tmin, float tmax, PrimHit* h, uint32_t* meta_out) {
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  float4 p0 = rec[0];
  uint32_t meta = meta_of(p0);
  *meta_out = meta;
  uint32_t kind = (meta >> GT_KIND_SHIFT) & GT_KIND_MASK;
  float4 p1 = rec[1];
  if (kind == GK_TRIANGLE) {
    float4 p2 = rec[2];
    return tri_hit(mk(p0.x, p0.y, p0.z), mk(p1.x, p1.y, p1.z), mk(p2.x, p2.y, p2.z), o, d, tmin, tmax, h);
  }
  if (kind == GK_QUAD) {
    float4 p2 = rec[2];
    float4 p3 = rec[3];
    return quad_hit(mk(p0.x, p0.y, p0.z), mk(p1.x, p1.y, p1.z), mk(p2.x, p2.y, p2.z), mk(p3.x, p3.y, p3.z), p1.w,
                    p2.w, p3.w, o, d, tmin, tmax, h);
  }
  f3 c = mk(p0.x, p0.y, p0.z);
  float r = p1.x;
  if (kind == GK_MOVING_SPHERE) {
    c = c + time * (mk(p1.x, p1.y, p1.z) - c);
    r = p1.w;
  }
  float root;
  if (!sphere_hit(c, r, o, d, tmin, tmax, &root)) return false;
  h->t = root; h->u = 0.f; h->v = 0.f;
  return true;
}
// ---- FP64 refinement of the chosen hit ---------------------------------------
// The FP32 traversal decides which primitive a ray hits. Its distance, and
// the surface coordinates, are then recomputed once per ray in FP64 with the
// reference's own expressions (contraction off, as the reference evaluates
// them): near the ray origin FP32 cannot resolve the distance to a surface
// (a ray 5 cm above the 1000-radius ground sphere loses 1e-3 of its t), FP64
// from the same FP32 inputs reproduces the reference's t to FP32 rounding.
// If FP64 rejects the primitive (an edge or silhouette case where the two
// precisions decide differently) the FP32 values stand.
struct d3 {
  double x, y, z;
};
__device__ __forceinline__ d3 dd(float4 v) { return {double(v.x), double(v.y), double(v.z)}; }
__device__ __forceinline__ d3 dd(f3 v) { return {double(v.x), double(v.y), double(v.z)}; }
__device__ __forceinline__ double ddot(d3 a, d3 b) {
#pragma clang fp contract(off)
  return a.x * b.x + a.y * b.y + a.z * b.z;
}
__device__ __forceinline__ d3 dsub(d3 a, d3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ d3 dcross(d3 a, d3 b) {
#pragma clang fp contract(off)
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ bool refine_hit(const GPrim* __restrict__ prims, uint32_t k, f3 of, f3 df, float time,
                                        float tmin, PrimHit* h) {
#pragma clang fp contract(off)
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  const float4 p0 = rec[0], p1 = rec[1];
  const uint32_t kind = (meta_of(p0) >> GT_KIND_SHIFT) & GT_KIND_MASK;
  const d3 o = dd(of), d = dd(df);
  const double lo = double(tmin);
  if (kind == GK_TRIANGLE) {  // geometry.rs:239-265
    const float4 p2 = rec[2];
    const d3 v0 = dd(p0), e1 = dd(p1), e2 = dd(p2);
    const d3 pv = dcross(d, e2);
    const double det = ddot(e1, pv);
    if (fabs(det) < 1e-10) return false;
    const double inv = 1.0 / det;
    const d3 tv = dsub(o, v0);
    const double u = ddot(tv, pv) * inv;
    if (!(u >= 0.0 && u <= 1.0)) return false;
    const d3 qv = dcross(tv, e1);
    const double v = ddot(d, qv) * inv;
    if (v < 0.0 || u + v > 1.0) return false;
    const double t = ddot(e2, qv) * inv;
    if (!(lo < t)) return false;
    h->t = float(t); h->u = float(u); h->v = float(v);
    return true;
  }
  if (kind == GK_QUAD) {  // QuadGeometry::new and hit_ray (geometry.rs:293-312,394-415)
    const float4 p2 = rec[2];
    const d3 c = dd(p0), u = dd(p1), v = dd(p2);
    const d3 n = dcross(u, v);
    const double nls = ddot(n, n);
    if (nls <= 2.220446049250313e-16) return false;
    const double len = sqrt(nls);
    const d3 nn = {n.x / len, n.y / len, n.z / len};
    const double pd = ddot(nn, c);
    const double denom = ddot(nn, d);
    if (fabs(denom) < 1e-8) return false;
    const double t = (pd - ddot(nn, o)) / denom;
    if (!(lo < t)) return false;
    const d3 w = {n.x / nls, n.y / nls, n.z / nls};
    const d3 pl = dsub({o.x + t * d.x, o.y + t * d.y, o.z + t * d.z}, c);
    const double a = ddot(w, dcross(pl, v)), b = ddot(w, dcross(u, pl));
    if (!(a >= 0.0 && a <= 1.0) || !(b >= 0.0 && b <= 1.0)) return false;
    h->t = float(t); h->u = float(a); h->v = float(b);
    return true;
  }
  // hit_sphere_in_interval (object.rs:986-1013): of the roots above t_min,
  // the one the FP32 test chose (the nearer to its distance)
  d3 c = dd(p0);
  double r = double(p1.x);
  if (kind == GK_MOVING_SPHERE) {  // geometry.rs:507-509
    const d3 c1 = dd(p1);
    const double tm = double(time);
    c = {c.x + tm * (c1.x - c.x), c.y + tm * (c1.y - c.y), c.z + tm * (c1.z - c.z)};
    r = double(p1.w);
  }
  const d3 oc = dsub(c, o);
  const double a = ddot(d, d);
  if (a <= 2.220446049250313e-16) return false;
  const double hh = ddot(d, oc);
  const double cc = ddot(oc, oc) - r * r;
  const double disc = hh * hh - a * cc;
  if (disc < 0.0) return false;
  const double sq = sqrt(disc);
  const double first = (hh - sq) / a, second = (hh + sq) / a;
  const double t32 = double(h->t);
  double t;
  if (lo < first && (!(lo < second) || fabs(first - t32) <= fabs(second - t32))) t = first;
  else if (lo < second) t = second;
  else return false;
  h->t = float(t);
  return true;
}

// Outward normal at a hit (object.rs:163-234); for spheres (p - c)/r, or the
// normalised offset when |r| <= EPS (geometry.rs:476-483).
__device__ __forceinline__ f3 prim_outward_normal(const GPrim* __restrict__ prims, uint32_t k, f3 p, float time,
                                                  uint32_t* material, uint32_t* kind_out) {
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  float4 p0 = rec[0];
  uint32_t meta = meta_of(p0);
  *material = meta & GT_MATERIAL_MASK;
  uint32_t kind = (meta >> GT_KIND_SHIFT) & GT_KIND_MASK;
  *kind_out = kind;
  if (kind == GK_TRIANGLE || kind == GK_QUAD) {
    float4 p3 = rec[3];
    return mk(p3.x, p3.y, p3.z);
  }
  float4 p1 = rec[1];
  f3 c = mk(p0.x, p0.y, p0.z);
  float r = p1.x;
  if (kind == GK_MOVING_SPHERE) {
    c = c + time * (mk(p1.x, p1.y, p1.z) - c);
    r = p1.w;
  }
  f3 out = p - c;
  if (fabsf(r) <= EPS) return normalized(out);
  return out / r;
}

// Shading normal of a mesh triangle (MeshTriangle::shading_normal,
// mesh.rs:105-119, oriented by set_shading_normal, object.rs:470-479): the
// vertex normals interpolated at barycentrics (u, v) of v1 and v2, normalized
// and flipped with the face; n itself (the oriented geometric normal) for a
// flat triangle, any other primitive, or a degenerate interpolation.
__device__ __forceinline__ f3 shading_normal(const GPrim* __restrict__ prims, const float4* __restrict__ vn,
                                             uint32_t k, float u, float v, bool front, f3 n) {
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  const float4 p1 = rec[1];
  const uint32_t kind = (meta_of(rec[0]) >> GT_KIND_SHIFT) & GT_KIND_MASK;
  const uint32_t smooth = __float_as_uint(p1.w);
  if (kind != GK_TRIANGLE || smooth == 0u) return n;
  const float4* q = vn + 3 * size_t(smooth - 1u);
  const float4 a = q[0], b = q[1], c = q[2];
  const float w = 1.0f - u - v;
  const f3 s = mk(w * a.x + u * b.x + v * c.x, w * a.y + u * b.y + v * c.y, w * a.z + u * b.z + v * c.z);
  if (!(len2(s) > EPS)) return n;
  const f3 sn = normalized(s);
  return front ? sn : -sn;
}
// Barycentric coordinates (of v1, v2) of a point p in a triangle record, for
// a hit whose FP64 refinement was rejected (an edge case).
__device__ __forceinline__ void tri_barycentric(const GPrim* __restrict__ prims, uint32_t k, f3 p, float* u,
                                                float* v) {
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  const float4 p0 = rec[0], p1 = rec[1], p2 = rec[2];
  const f3 e1 = mk(p1.x, p1.y, p1.z), e2 = mk(p2.x, p2.y, p2.z), q = p - mk(p0.x, p0.y, p0.z);
  const float d00 = dot(e1, e1), d01 = dot(e1, e2), d11 = dot(e2, e2), d20 = dot(q, e1), d21 = dot(q, e2);
  const float den = d00 * d11 - d01 * d01;
  if (!(fabsf(den) > 0.f)) { *u = 0.f; *v = 0.f; return; }
  *u = (d11 * d20 - d01 * d21) / den;
  *v = (d00 * d21 - d01 * d20) / den;
}

// ---- scene and traversal ---------------------------------------------------
struct DScene {
  const GNode2* __restrict__ nodes2;
  const GNode4* __restrict__ nodes4;
  const GPrim* __restrict__ prims;
  const float4* __restrict__ vnormals;  // mesh triangles' vertex normals, 3 per triangle
  const uint32_t* __restrict__ prim_ids;
  const GMat* __restrict__ mats;
  float root_lo[3], root_hi[3];
  uint32_t root_ref;
  uint32_t width;  // 2 or 4
};

struct Stats {
  uint32_t node_tests, node_hits, leaf_visits, candidates, leaf_hits, max_stack;
};

// Per-lane traversal stack: the first `cap` entries in LDS (lane-interleaved),
// the rest in a per-lane slice of global memory. Each part is reached through a
// pointer of its own address space: through a common one the compiler merges
// the two accesses into flat instructions, which occupy the vector memory path
// and both wait counters for what is nearly always an LDS access.
typedef uint32_t stack_entry __attribute__((ext_vector_type(2)));  // child reference, entry distance
typedef __attribute__((address_space(3))) stack_entry lds_entry;
typedef __attribute__((address_space(1))) stack_entry global_entry;
struct Stack {
  uint32_t lds;     // LDS address of the lane's first entry
  uint32_t stride;  // bytes between a lane's entries
  global_entry* glob;
  uint32_t gstride;
  int cap;
  int n;
  __device__ __forceinline__ lds_entry* slot() const { return (lds_entry*)(__umul24(n, stride) + lds); }
  __device__ __forceinline__ global_entry* spill() const { return glob + size_t(uint32_t(n - cap)) * gstride; }
  __device__ __forceinline__ void push(uint32_t ref, float t) {
    const stack_entry e = {ref, __float_as_uint(t)};
    if (__ballot(n >= cap) == 0ull) {  // the usual case for every lane
      *slot() = e;
    } else {
      if (n < cap) *slot() = e;
      else *spill() = e;
    }
    ++n;
  }
  __device__ __forceinline__ uint2 pop() {
    --n;
    stack_entry e;
    if (__ballot(n >= cap) == 0ull) {
      e = *slot();
    } else {
      if (n < cap) e = *slot();
      else e = *spill();
    }
    return make_uint2(e.x, e.y);
  }
};

// Precomputed slab data (RayTraversal::new, bvh.rs:98-117). A parallel axis
// (|d| <= EPS) gets inv = +inf, which with IEEE maxNum/minNum reproduces the
// reference's origin-in-slab rule: (lo-o)*inf is -inf, +inf or NaN (ignored).
struct RayPre {
  f3 o;
  float inv[3];
  bool neg[3];
};
__device__ __forceinline__ RayPre ray_pre(f3 o, f3 d) {
  RayPre r;
  r.o = o;
  float dd[3] = {d.x, d.y, d.z};
  const bool plain = beyond_rcp(fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z)));
  for (int a = 0; a < 3; ++a) {
    bool par = fabsf(dd[a]) <= EPS;
    r.inv[a] = par ? INF : plain ? 1.0f / dd[a] : rcp_rn(dd[a]);
    r.neg[a] = r.inv[a] < 0.f;
  }
  return r;
}
// Slab test, conservative in FP32 (the far bound is widened by a few ulp);
// returns the entry distance or -1 for a miss.
__device__ __forceinline__ bool slab(const RayPre& r, float lox, float hix, float loy, float hiy, float loz, float hiz,
                                     float tmin, float tmax, float* entry) {
  float nx = r.neg[0] ? hix : lox, fx = r.neg[0] ? lox : hix;
  float ny = r.neg[1] ? hiy : loy, fy = r.neg[1] ? loy : hiy;
  float nz = r.neg[2] ? hiz : loz, fz = r.neg[2] ? loz : hiz;
  float t0x = (nx - r.o.x) * r.inv[0], t1x = (fx - r.o.x) * r.inv[0];
  float t0y = (ny - r.o.y) * r.inv[1], t1y = (fy - r.o.y) * r.inv[1];
  float t0z = (nz - r.o.z) * r.inv[2], t1z = (fz - r.o.z) * r.inv[2];
  float en = fmaxf(fmaxf(tmin, t0x), fmaxf(t0y, t0z));
  float ex = fminf(fminf(tmax, t1x), fminf(t1y, t1z));
  *entry = en;
  return ex * 1.0000004f >= en;
}

// Closest hit over the BVH2 layout, walking the reference's order: both children tested against the current
// closest, nearer first (left on ties), entries pruned when entry >= closest
// (bvh.rs:306-399). Leaves test primitives in permutation order with the
// interval shrinking on each accepted hit (scene.rs:849-874).
template <bool STATS>
__device__ __forceinline__ bool trace2(const DScene& sc, f3 o, f3 d, float time, float tmin, float tmax,
                                       Stack& st, float* t_out, uint32_t* prim_out, PrimHit* hit_out, Stats* stats) {
  RayPre rp = ray_pre(o, d);
  float closest = tmax;
  bool any = false;
  uint32_t best = 0;
  PrimHit bh{0.f, 0.f, 0.f};
  if (STATS) { stats->node_tests += 1; }
  float root_entry;
  if (!slab(rp, sc.root_lo[0], sc.root_hi[0], sc.root_lo[1], sc.root_hi[1], sc.root_lo[2], sc.root_hi[2], tmin,
            tmax, &root_entry))
    return false;
  if (STATS) { stats->node_hits += 1; stats->max_stack = max(stats->max_stack, 1u); }
  uint32_t cur = sc.root_ref;
  st.n = 0;
  for (;;) {
    if (cur & GT_LEAF_BIT) {
      uint32_t k = cur & ~GT_LEAF_BIT;
      bool leaf_hit = false;
      if (STATS) stats->leaf_visits += 1;
      for (;;) {
        PrimHit h;
        uint32_t meta;
        if (STATS) stats->candidates += 1;
        if (prim_test(sc.prims, k, o, d, time, tmin, closest, &h, &meta)) {
          closest = h.t;
          best = k;
          bh = h;
          any = true;
          leaf_hit = true;
        }
        if (meta & GT_LAST_BIT) break;
        ++k;
      }
      if (STATS && leaf_hit) stats->leaf_hits += 1;
    } else {
      const float4* nd = reinterpret_cast<const float4*>(sc.nodes2 + cur);
      float4 a = nd[0], b = nd[1], c = nd[2];
      uint4 refs = *reinterpret_cast<const uint4*>(nd + 3);
      float le, re;
      bool lh = slab(rp, a.x, a.y, a.z, a.w, c.x, c.y, tmin, closest, &le);
      bool rh = slab(rp, b.x, b.y, b.z, b.w, c.z, c.w, tmin, closest, &re);
      if (STATS) {
        stats->node_tests += 2;
        stats->node_hits += uint32_t(lh) + uint32_t(rh);
        uint32_t len = uint32_t(st.n) + uint32_t(lh) + uint32_t(rh);
        stats->max_stack = max(stats->max_stack, len);
      }
      if (lh && rh) {
        bool right_first = re < le;
        uint32_t nearer = right_first ? refs.y : refs.x;
        uint32_t farther = right_first ? refs.x : refs.y;
        st.push(farther, right_first ? le : re);
        cur = nearer;
        continue;
      }
      if (lh) { cur = refs.x; continue; }
      if (rh) { cur = refs.y; continue; }
    }
    // pop, skipping entries that cannot beat the current closest hit
    bool found = false;
    while (st.n > 0) {
      uint2 e = st.pop();
      if (__uint_as_float(e.y) >= closest) continue;
      cur = e.x;
      found = true;
      break;
    }
    if (!found) break;
  }
  if (any) {
    *t_out = closest;
    *prim_out = best;
    if (hit_out) *hit_out = bh;
  }
  return any;
}

// Four-wide variant: children of a wide node are visited nearest-first.
template <bool STATS>
__device__ __forceinline__ bool trace4(const DScene& sc, f3 o, f3 d, float time, float tmin, float tmax,
                                       Stack& st, float* t_out, uint32_t* prim_out, PrimHit* hit_out, Stats* stats) {
  RayPre rp = ray_pre(o, d);
  float closest = tmax;
  bool any = false;
  uint32_t best = 0;
  PrimHit bh{0.f, 0.f, 0.f};
  float root_entry;
  if (STATS) stats->node_tests += 1;
  if (!slab(rp, sc.root_lo[0], sc.root_hi[0], sc.root_lo[1], sc.root_hi[1], sc.root_lo[2], sc.root_hi[2], tmin,
            tmax, &root_entry))
    return false;
  if (STATS) { stats->node_hits += 1; stats->max_stack = max(stats->max_stack, 1u); }
  uint32_t cur = sc.root_ref;
  st.n = 0;
  for (;;) {
    if (cur & GT_LEAF_BIT) {
      uint32_t k = cur & ~GT_LEAF_BIT;
      bool leaf_hit = false;
      if (STATS) stats->leaf_visits += 1;
      for (;;) {
        PrimHit h;
        uint32_t meta;
        if (STATS) stats->candidates += 1;
        if (prim_test(sc.prims, k, o, d, time, tmin, closest, &h, &meta)) {
          closest = h.t; best = k; bh = h; any = true; leaf_hit = true;
        }
        if (meta & GT_LAST_BIT) break;
        ++k;
      }
      if (STATS && leaf_hit) stats->leaf_hits += 1;
    } else {
      const float4* nd = reinterpret_cast<const float4*>(sc.nodes4 + cur);
      float4 lox = nd[0], hix = nd[1], loy = nd[2], hiy = nd[3], loz = nd[4], hiz = nd[5];
      uint4 ch = *reinterpret_cast<const uint4*>(nd + 6);
      float e[4];
      bool h[4];
      h[0] = slab(rp, lox.x, hix.x, loy.x, hiy.x, loz.x, hiz.x, tmin, closest, &e[0]) && ch.x != GT_EMPTY_CHILD;
      h[1] = slab(rp, lox.y, hix.y, loy.y, hiy.y, loz.y, hiz.y, tmin, closest, &e[1]) && ch.y != GT_EMPTY_CHILD;
      h[2] = slab(rp, lox.z, hix.z, loy.z, hiy.z, loz.z, hiz.z, tmin, closest, &e[2]) && ch.z != GT_EMPTY_CHILD;
      h[3] = slab(rp, lox.w, hix.w, loy.w, hiy.w, loz.w, hiz.w, tmin, closest, &e[3]) && ch.w != GT_EMPTY_CHILD;
      uint32_t c[4] = {ch.x, ch.y, ch.z, ch.w};
      if (STATS) {
        stats->node_tests += 4;
        stats->node_hits += uint32_t(h[0]) + uint32_t(h[1]) + uint32_t(h[2]) + uint32_t(h[3]);
      }
      // order hit children by entry (stable: lower slot first on ties), push
      // all but the nearest in far-to-near order
      int idx[4];
      int nh = 0;
      for (int k = 0; k < 4; ++k) if (h[k]) idx[nh++] = k;
      for (int i = 1; i < nh; ++i) {
        int v = idx[i];
        int j = i - 1;
        while (j >= 0 && e[idx[j]] > e[v]) { idx[j + 1] = idx[j]; --j; }
        idx[j + 1] = v;
      }
      if (STATS) stats->max_stack = max(stats->max_stack, uint32_t(st.n + nh));
      if (nh > 0) {
        for (int i = nh - 1; i >= 1; --i) st.push(c[idx[i]], e[idx[i]]);
        cur = c[idx[0]];
        continue;
      }
    }
    bool found = false;
    while (st.n > 0) {
      uint2 en = st.pop();
      if (__uint_as_float(en.y) >= closest) continue;
      cur = en.x;
      found = true;
      break;
    }
    if (!found) break;
  }
  if (any) {
    *t_out = closest;
    *prim_out = best;
    if (hit_out) *hit_out = bh;
  }
  return any;
}

template <bool STATS>
__device__ __forceinline__ bool trace(const DScene& sc, f3 o, f3 d, float time, float tmin, float tmax, Stack& st,
                                      float* t_out, uint32_t* prim_out, PrimHit* hit_out, Stats* stats) {
  if (sc.width == 4) return trace4<STATS>(sc, o, d, time, tmin, tmax, st, t_out, prim_out, hit_out, stats);
  return trace2<STATS>(sc, o, d, time, tmin, tmax, st, t_out, prim_out, hit_out, stats);
}

// ---- resumable walk -----------------------------------------------------------
// The same search as trace, one step at a time: the state of a ray between
// steps, so that a wave can mix rays at different points of their walks. A
// ray's steps (nodes fetched, primitives tested, the closest hit each is tested
// against) are those of trace2 / trace4, in the same order, whatever the other
// lanes do. tmin is SHADOW_ACNE and the interval starts unbounded.
constexpr uint32_t kNoNode = 0xffffffffu;  // walk over (has the leaf bit; no leaf has this index)
constexpr uint32_t kNoPrim = 0xffffffffu;
constexpr uint32_t kNoSelf = 0xffffffffu;  // a camera ray starts on no primitive
struct Walk {
  f3 o, d;
  float inv[3];
  float rdd;     // 1 / |d|^2
  float time, closest;
  uint32_t cur;  // node, GT_LEAF_BIT | primitive, or kNoNode
  uint32_t self, best;  // primitives (leaf order): where the ray starts (or kNoSelf), the closest hit (or kNoPrim)
};
// The scene's part that the steps read, with pointers known to be global.
struct WalkScene {
  const float4* nodes;  // GNode2 or GNode4 records
  const GPrim* prims;
};
template <bool WIDE>
__device__ __forceinline__ WalkScene walk_scene(const DScene& sc) {
  return {WIDE ? reinterpret_cast<const float4*>(sc.nodes4) : reinterpret_cast<const float4*>(sc.nodes2),
          sc.prims};
}
// The stack's bottom entry ends the walk, so a pop needs no test for an empty stack.
__device__ __forceinline__ void walk_begin(const DScene& sc, f3 o, f3 d, float time, uint32_t self, Walk& w, Stack& st) {
  const RayPre rp = ray_pre(o, d);
  w.o = o;
  w.d = d;
  for (int a = 0; a < 3; ++a) w.inv[a] = rp.inv[a];
  w.rdd = reciprocal(len2(d));
  w.time = time;
  w.closest = INF;
  w.self = self;
  w.best = kNoPrim;
  st.n = 0;
  st.push(kNoNode, -INF);
  float entry;
  w.cur = slab(rp, sc.root_lo[0], sc.root_hi[0], sc.root_lo[1], sc.root_hi[1], sc.root_lo[2], sc.root_hi[2],
               SHADOW_ACNE, INF, &entry)
              ? sc.root_ref
              : kNoNode;
}
// The next stack entry that can beat the closest hit, or kNoNode.
__device__ __forceinline__ uint32_t walk_pop(float closest, Stack& st) {
  uint2 e;
  do e = st.pop();
  while (!(__uint_as_float(e.y) < closest));
  return e.x;
}
// One inner node: w.cur is a node index.
template <bool WIDE>
__device__ __forceinline__ void walk_inner(const WalkScene& sc, Walk& w, Stack& st) {
  RayPre rp;
  rp.o = w.o;
  for (int a = 0; a < 3; ++a) { rp.inv[a] = w.inv[a]; rp.neg[a] = w.inv[a] < 0.f; }
  if (!WIDE) {
    const float4* nd = sc.nodes + 4 * size_t(w.cur);
    const float4 a = nd[0], b = nd[1], c = nd[2];
    const uint2 refs = *reinterpret_cast<const uint2*>(nd + 3);
    float le, re;
    const bool lh = slab(rp, a.x, a.y, a.z, a.w, c.x, c.y, SHADOW_ACNE, w.closest, &le);
    const bool rh = slab(rp, b.x, b.y, b.z, b.w, c.z, c.w, SHADOW_ACNE, w.closest, &re);
    const bool nearer = re < le;
    const bool right = lh ? nearer : true;  // the nearer child, left on ties
    const bool r = rh ? right : false;
    const bool both = lh ? rh : false, none = lh ? false : !rh;
    w.cur = r ? refs.y : refs.x;
    if (both) st.push(r ? refs.x : refs.y, r ? le : re);
    if (none) w.cur = walk_pop(w.closest, st);
    return;
  }
  const float4* nd = sc.nodes + 8 * size_t(w.cur);
  const float4 lox = nd[0], hix = nd[1], loy = nd[2], hiy = nd[3], loz = nd[4], hiz = nd[5];
  const uint4 ch = *reinterpret_cast<const uint4*>(nd + 6);
  float e[4];
  bool h[4];
  h[0] = slab(rp, lox.x, hix.x, loy.x, hiy.x, loz.x, hiz.x, SHADOW_ACNE, w.closest, &e[0]) && ch.x != GT_EMPTY_CHILD;
  h[1] = slab(rp, lox.y, hix.y, loy.y, hiy.y, loz.y, hiz.y, SHADOW_ACNE, w.closest, &e[1]) && ch.y != GT_EMPTY_CHILD;
  h[2] = slab(rp, lox.z, hix.z, loy.z, hiy.z, loz.z, hiz.z, SHADOW_ACNE, w.closest, &e[2]) && ch.z != GT_EMPTY_CHILD;
  h[3] = slab(rp, lox.w, hix.w, loy.w, hiy.w, loz.w, hiz.w, SHADOW_ACNE, w.closest, &e[3]) && ch.w != GT_EMPTY_CHILD;
  const uint32_t c[4] = {ch.x, ch.y, ch.z, ch.w};
  // as trace4: hit children by entry (lower slot first on ties), all but the nearest pushed far to near
  int idx[4];
  int nh = 0;
  for (int k = 0; k < 4; ++k) if (h[k]) idx[nh++] = k;
  for (int i = 1; i < nh; ++i) {
    int v = idx[i];
    int j = i - 1;
    while (j >= 0 && e[idx[j]] > e[v]) { idx[j + 1] = idx[j]; --j; }
    idx[j + 1] = v;
  }
  if (nh > 0) {
    for (int i = nh - 1; i >= 1; --i) st.push(c[idx[i]], e[idx[i]]);
    w.cur = c[idx[0]];
  } else {
    w.cur = walk_pop(w.closest, st);
  }
}
// prim_test's decision and distance, with the tests of a kind in one straight line: a wave takes
// every path some lane needs, so early exits save nothing, and sphere_hit's quotients share 1 / |d|^2.
//
// self: the ray starts on this primitive. A ray leaving a plane cannot meet it again (the reference's t
// is 0 up to rounding, below t_min). On a sphere one root is then 0 in exact arithmetic and the other
// 2h/a, so it is met again only by a ray heading inward, at the far root. FP32 cannot place the origin
// on a large sphere within t_min (on the 1000-radius ground sphere a coordinate's ulp is 6e-5 and the
// near root's error grows as 1/cos at grazing angles), so the near root is skipped by this rule, not
// compared with t_min: the decision the reference's f64 arithmetic makes.
__device__ __forceinline__ bool walk_test(const GPrim* __restrict__ prims, uint32_t k, const Walk& w, float* t_out,
                                          uint32_t* meta_out) {
  const float4* rec = reinterpret_cast<const float4*>(prims + k);
  const float4 p0 = rec[0], p1 = rec[1];
  const uint32_t meta = meta_of(p0);
  *meta_out = meta;
  const uint32_t kind = (meta >> GT_KIND_SHIFT) & GT_KIND_MASK;
  const bool self = k == w.self;
  const float tmin = SHADOW_ACNE, tmax = w.closest;
  if (kind == GK_TRIANGLE) {  // tri_hit
    const float4 p2 = rec[2];
    const f3 e1 = mk(p1.x, p1.y, p1.z), e2 = mk(p2.x, p2.y, p2.z);
    const f3 pvec = cross(w.d, e2);
    const float det = dot(e1, pvec);
    const float inv = reciprocal(det);
    const f3 tvec = w.o - mk(p0.x, p0.y, p0.z);
    const float u = dot(tvec, pvec) * inv;
    const f3 qvec = cross(tvec, e1);
    const float v = dot(w.d, qvec) * inv;
    const float t = dot(e2, qvec) * inv;
    *t_out = t;
    return !(fabsf(det) < 1e-10f) & (u >= 0.f) & (u <= 1.f) & !(v < 0.f) & !(u + v > 1.f) & (tmin < t) & (t < tmax) & !self;
  }
  if (kind == GK_QUAD) {  // quad_hit
    const float4 p2 = rec[2], p3 = rec[3];
    const f3 n = mk(p3.x, p3.y, p3.z);
    const float denom = dot(n, w.d);
    const float t = (p3.w - dot(n, w.o)) / denom;
    const f3 pp = (w.o + t * w.d) - mk(p0.x, p0.y, p0.z);
    const f3 wn = n * p1.w;
    const float u = dot(wn, cross(pp, mk(p2.x, p2.y, p2.z))), v = dot(wn, cross(mk(p1.x, p1.y, p1.z), pp));
    *t_out = t;
    return !(p2.w <= EPS) & !(fabsf(denom) < 1e-8f) & (tmin < t) & (t < tmax) & (u >= 0.f) & (u <= 1.f) & (v >= 0.f) &
           (v <= 1.f) & !self;
  }
  f3 c = mk(p0.x, p0.y, p0.z);
  float r = p1.x;
  if (kind == GK_MOVING_SPHERE) {
    c = c + w.time * (mk(p1.x, p1.y, p1.z) - c);
    r = p1.w;
  }
  const f3 oc = c - w.o;  // sphere_hit
  const float a = len2(w.d);
  const float h = dot(w.d, oc);
  const f3 perp = oc - div_rn(h, a, w.rdd) * w.d;
  const float disc = a * (r * r - len2(perp));
  if (a <= EPS || disc < 0.f || (self && h <= 0.f)) return false;
  const float sq = sqrt_rn(disc);
  const float first = div_rn(h - sq, a, w.rdd), second = div_rn(h + sq, a, w.rdd);
  const bool near_root = !self && tmin < first && first < tmax;
  *t_out = near_root ? first : second;
  return near_root || (tmin < second && second < tmax);
}
// One primitive of a leaf: w.cur is GT_LEAF_BIT | its index. With ANY the first hit ends the walk.
template <bool ANY>
__device__ __forceinline__ void walk_leaf(const WalkScene& sc, Walk& w, Stack& st) {
  const uint32_t k = w.cur & ~GT_LEAF_BIT;
  float t;
  uint32_t meta;
  const bool hit = walk_test(sc.prims, k, w, &t, &meta);
  if (hit) {
    w.closest = t;
    w.best = k;
  }
  const bool over = ANY && hit, last = (meta & GT_LAST_BIT) != 0u;
  w.cur = over ? kNoNode : w.cur + 1;
  if (last && !over) w.cur = walk_pop(w.closest, st);
}

// ---- light targets (scene.rs:363-609, object.rs:1048-1161) --------------------
struct DLights {
  const GLight* __restrict__ l;
  uint32_t n;
  float total;
};
__device__ __forceinline__ float area_pdf(f3 dir, float t, f3 n, float area) {  // object.rs:1101-1113
  if (area <= EPS) return 0.f;
  float d2 = len2(t * dir);
  float cosine = fabsf(dot(normalized(dir), n));
  if (cosine <= EPS) return 0.f;
  return d2 / (cosine * area);
}
__device__ __forceinline__ float light_pdf_one(const GLight& L, f3 origin, float time, f3 dir) {
  uint32_t kind = uint32_t(L.c[3]);
  if (kind == GK_SPHERE || kind == GK_MOVING_SPHERE) {  // object.rs:1048-1073
    f3 c = ld3(L.a);
    if (kind == GK_MOVING_SPHERE) c = c + time * (ld3(L.b) - c);
    float r = L.a[3];
    float root;
    if (!sphere_hit(c, r, origin, dir, SHADOW_ACNE, INF, &root)) return 0.f;
    float d2 = len2(c - origin);
    float r2 = r * r;
    if (d2 <= r2) return 1.0f / (4.0f * PI);
    float cos_max = sqrt_rn(1.0f - r2 / d2);
    float sa = 2.0f * PI * (1.0f - cos_max);
    return sa <= EPS ? 0.f : 1.0f / sa;
  }
  PrimHit h;
  if (kind == GK_TRIANGLE) {
    if (!tri_hit(ld3(L.a), ld3(L.b), ld3(L.c), origin, dir, SHADOW_ACNE, INF, &h)) return 0.f;
  } else {
    if (!quad_hit(ld3(L.a), ld3(L.b), ld3(L.c), ld3(L.n), L.w[0], L.w[1], L.w[3], origin, dir, SHADOW_ACNE, INF, &h))
      return 0.f;
  }
  return area_pdf(dir, h.t, ld3(L.n), L.n[3]);
}
__device__ __forceinline__ float lights_pdf(const DLights& ls, f3 origin, float time, f3 dir) {  // scene.rs:571-582
  if (ls.n == 0 || ls.total <= 0.f) return 0.f;
  float sum = 0.f;
  for (uint32_t i = 0; i < ls.n; ++i) sum += ls.l[i].b[3] * light_pdf_one(ls.l[i], origin, time, dir);
  return sum;
}
__device__ __forceinline__ f3 light_random_one(const GLight& L, f3 origin, float time, Rng& rng) {
  uint32_t kind = uint32_t(L.c[3]);
  if (kind == GK_SPHERE || kind == GK_MOVING_SPHERE) {  // object.rs:1115-1130
    f3 c = ld3(L.a);
    if (kind == GK_MOVING_SPHERE) c = c + time * (ld3(L.b) - c);
    float r = L.a[3];
    f3 dir = c - origin;
    float d2 = len2(dir);
    float r2 = r * r;
    if (d2 <= r2 || d2 <= EPS) return rng.unit_vector_spherical();
    float r1 = rng.next(), rr2 = rng.next();  // random_to_sphere :1154-1161
    float z = 1.0f + rr2 * (sqrt_rn(1.0f - r2 / d2) - 1.0f);
    float phi = 2.0f * PI * r1;
    float rz = sqrt_rn(1.0f - z * z);
    float s, cc;
    sincosf(phi, &s, &cc);
    f3 local = mk(cc * rz, s * rz, z);
    Onb b;
    return onb_from_w(dir, &b) ? b.local(local) : local;
  }
  if (kind == GK_TRIANGLE) {  // :1138-1152
    float a = rng.next();
    float b = rng.next();
    if (a + b > 1.0f) { a = 1.0f - a; b = 1.0f - b; }
    f3 p = ld3(L.a) + a * ld3(L.b) + b * ld3(L.c);
    return p - origin;
  }
  float a = rng.next();  // quad :1132-1136
  f3 p0 = ld3(L.a) + a * ld3(L.b);
  float b = rng.next();
  return (p0 + b * ld3(L.c)) - origin;
}
__device__ __forceinline__ f3 lights_random(const DLights& ls, f3 origin, float time, Rng& rng) {  // scene.rs:584-600
  if (ls.n == 0 || ls.total <= 0.f) return mk(1.f, 0.f, 0.f);
  float pick = rng.range(0.f, ls.total);
  for (uint32_t i = 0; i < ls.n; ++i) {
    pick -= ls.l[i].w[2];  // raw weight
    if (pick <= 0.f) return light_random_one(ls.l[i], origin, time, rng);
  }
  return light_random_one(ls.l[ls.n - 1], origin, time, rng);
}

// ---- environment (environment.rs) ---------------------------------------------
struct DEnv {
  uint32_t kind;        // 0 none, 1 constant, 2 texture
  uint32_t w, h;
  uint32_t uniform;     // total weight <= EPS: uniform sphere sampling
  float color[3];
  // Linear RGB texels, row-major, row 0 at +y; .w holds the texel's
  // solid-angle pdf (:136-156), so a pdf lookup shares the cache line of the
  // radiance lookup around the same direction.
  const float4* __restrict__ tex;
  // Alias table over the texels (Vose's method): slot i keeps texel i when
  // the low 32 bits of its draw are below .x and otherwise yields texel .y.
  // It samples the reference's texel distribution (rebuild_distribution,
  // :158-184) with one draw and two dependent loads instead of a search.
  const uint2* __restrict__ alias;
  // cos of the polar angle of each row's edges (h + 1 values, made by env_row_cos), and what
  // splits a texel index into row and column
  const float* __restrict__ row_cos;
  Div31 row;
  float inv_w;  // 1 / w
};
// The polar angle's cosine at the upper edge of row y.
__device__ __forceinline__ float env_row_cos(uint32_t y, uint32_t h) { return cosf(PI * (float(y) / float(h))); }
__device__ __forceinline__ float power_heuristic(float a, float b) {  // camera.rs:2486-2496
  if (!isfinite(a) || a <= EPS) return 0.f;
  if (!isfinite(b) || b <= EPS) return 1.0f;
  float s = a * a, o = b * b;
  return s / (s + o);
}
// rem_euclid of an angle in [-TAU, TAU) by TAU, and of a coordinate in [0, 2) by 1: the
// remainder itself is exact, so these are fmodf's values without its loop.
__device__ __forceinline__ float wrap_angle(float phi) { return phi < 0.f ? phi + TAU : phi; }
__device__ __forceinline__ float wrap_unit(float u) { return u >= 1.0f ? u - 1.0f : u; }
__device__ __forceinline__ f3 env_radiance_uv(const DEnv& e, float u, float v);
__device__ __forceinline__ f3 env_radiance(const DEnv& e, f3 dir) {  // :98-107
  if (e.kind == 1) return ld3(e.color);
  f3 d = normalized(dir);
  float phi = wrap_angle(atan2f(d.z, d.x));
  float theta = acosf(clampf(d.y, -1.f, 1.f));
  float u = div_rn(phi, TAU, INV_TAU), v = 1.0f - div_rn(theta, PI, INV_PI);
  if (!isfinite(u) || !isfinite(v)) return mk(0.f, 0.f, 0.f);
  return env_radiance_uv(e, u, v);
}
// pdf_value (:136-156) of a direction at lat-long angles (phi, theta): the
// solid-angle pdf of the texel that holds it.
__device__ __forceinline__ float env_pdf_at(const DEnv& e, float phi, float theta) {
  if (e.kind != 2 || e.uniform) return 1.0f / (4.0f * PI);
  float fx = floorf(div_rn(phi, TAU, INV_TAU) * float(e.w)), fy = floorf(div_rn(theta, PI, INV_PI) * float(e.h));
  uint32_t x = fx > 0.f ? min(uint32_t(fx), e.w - 1) : 0u;
  uint32_t y = fy > 0.f ? min(uint32_t(fy), e.h - 1) : 0u;
  return e.tex[size_t(y) * e.w + x].w;
}
// env_radiance(dir) for a path that missed. On entry *mw is the path's MIS
// weight, or -cpdf when the weight is the environment's power heuristic
// power_heuristic(cpdf, pdf_value(dir)); on return it is the weight. The
// direction maps to lat-long coordinates once for both lookups.
__device__ __forceinline__ f3 env_radiance_weighted(const DEnv& e, f3 dir, float* mw) {
  if (e.kind != 2) {
    if (*mw < 0.f) *mw = power_heuristic(-*mw, env_pdf_at(e, 0.f, 0.f));
    return ld3(e.color);
  }
  f3 d = normalized(dir);
  float phi = wrap_angle(atan2f(d.z, d.x));
  float theta = acosf(clampf(d.y, -1.f, 1.f));
  if (*mw < 0.f) *mw = power_heuristic(-*mw, env_pdf_at(e, phi, theta));
  float u = div_rn(phi, TAU, INV_TAU), v = 1.0f - div_rn(theta, PI, INV_PI);
  if (!isfinite(u) || !isfinite(v)) return mk(0.f, 0.f, 0.f);
  return env_radiance_uv(e, u, v);
}
// The sampled texel's radiance and pdf. The reference evaluates
// pdf_value(direction) and radiance(direction) from the returned direction
// (environment.rs:130-131); the direction lies in texel (x, y) by
// construction, so the texel's pdf and the lat-long coordinates
// u = (x + r) / w, theta = acos(cos theta) are used directly.
struct EnvSample {
  f3 dir;
  float pdf;
  float u, cos_theta;
  bool texel;
};
__device__ __forceinline__ f3 env_radiance_uv(const DEnv& e, float u, float v) {  // texture.rs:681-711
  float cx = wrap_unit(u) * float(e.w);
  uint32_t x0 = min(uint32_t(floorf(cx)), e.w - 1);
  uint32_t x1 = (x0 + 1 == e.w) ? 0 : x0 + 1;
  float cy = clampf(1.0f - v, 0.f, 1.f) * float(e.h - 1);
  uint32_t y0 = min(uint32_t(floorf(cy)), e.h - 1);
  uint32_t y1 = min(y0 + 1, e.h - 1);
  float tx = cx - float(x0), ty = cy - float(y0);
  const float4* tex = e.tex;
  float4 a = tex[size_t(y0) * e.w + x0], b = tex[size_t(y0) * e.w + x1];
  float4 c = tex[size_t(y1) * e.w + x0], f = tex[size_t(y1) * e.w + x1];
  f3 top = mk(a.x + (b.x - a.x) * tx, a.y + (b.y - a.y) * tx, a.z + (b.z - a.z) * tx);
  f3 bot = mk(c.x + (f.x - c.x) * tx, c.y + (f.y - c.y) * tx, c.z + (f.z - c.z) * tx);
  return top + (bot - top) * ty;
}
__device__ __forceinline__ EnvSample env_sample(const DEnv& e, Rng& rng) {  // :109-132
  EnvSample r;
  if (e.kind != 2 || e.uniform) {
    r.dir = rng.unit_vector_spherical();
    r.pdf = 1.0f / (4.0f * PI);
    r.texel = false;
    return r;
  }
  // The texel: slot = floor(draw * n) from the high bits of draw * n, the
  // keep-or-alias test from its low bits (one 64-bit draw, integer math).
  const uint64_t draw = rng.next_u64();
  const uint64_t n = uint64_t(e.w) * e.h;
  const uint32_t slot = uint32_t(__umul64hi(draw, n));
  const uint32_t frac = uint32_t((draw * n) >> 32);
  const uint2 rec = e.alias[slot];
  const uint32_t texel = frac < rec.x ? slot : rec.y;
  uint32_t x;
  const uint32_t y = div31(texel, e.row, &x);
  float u = div_rn(float(x) + rng.next(), float(e.w), e.inv_w);
  const float c0 = e.row_cos[y], c1 = e.row_cos[y + 1];
  float ct = c0 + rng.next() * (c1 - c0);
  float st = sqrt_rn(fmaxf(1.0f - ct * ct, 0.f));
  float phi = TAU * u;
  float s, c;
  sincosf(phi, &s, &c);
  r.dir = mk(st * c, ct, st * s);
  r.pdf = e.tex[size_t(y) * e.w + x].w;
  r.u = u;
  r.cos_theta = ct;
  r.texel = true;
  return r;
}
__device__ __forceinline__ f3 env_sample_radiance(const DEnv& e, const EnvSample& s) {
  if (e.kind == 1) return ld3(e.color);
  if (!s.texel) return env_radiance(e, s.dir);
  float theta = acosf(clampf(s.cos_theta, -1.f, 1.f));
  return env_radiance_uv(e, s.u, 1.0f - div_rn(theta, PI, INV_PI));
}


// ---- camera rays (camera.rs:1658-1718) ------------------------------------------
__device__ __forceinline__ void camera_ray(const GCamera& cam, uint32_t x, uint32_t y, uint32_t s, Rng& rng, f3* o,
                                           f3* d, float* time) {
  float ox, oy;
  if (cam.mode == 0) {
    ox = rng.next() - 0.5f;
    oy = rng.next() - 0.5f;
  } else {
    uint32_t sx = s % cam.grid, sy = s / cam.grid;
    float rec = 1.0f / float(cam.grid);
    ox = ((float(sx) + rng.next()) * rec) - 0.5f;
    oy = ((float(sy) + rng.next()) * rec) - 0.5f;
  }
  f3 ps = ld3(cam.pixel00) + (float(x) + ox) * ld3(cam.du) + (float(y) + oy) * ld3(cam.dv);
  f3 origin = ld3(cam.center);
  if (cam.defocus) {
    f3 dk = rng.in_unit_disk();
    origin = origin + dk.x * ld3(cam.disk_u) + dk.y * ld3(cam.disk_v);
  }
  *time = rng.range(cam.shutter_start, cam.shutter_end);
  *o = origin;
  *d = ps - origin;
}
__device__ __forceinline__ f3 background(const GCamera& cam, f3 dir) {  // camera.rs:297-313
  if (cam.background_kind == 1) {
    f3 nadir = ld3(cam.background), horizon = ld3(cam.background + 3), zenith = ld3(cam.background + 6);
    float t = 0.5f * (normalized(dir).y + 1.0f);
    if (t < 0.5f) { float bl = 2.0f * t; return nadir * (1.0f - bl) + horizon * bl; }
    float bl = 2.0f * (t - 0.5f);
    return horizon * (1.0f - bl) + zenith * bl;
  }
  return ld3(cam.background);
}

}  // namespace gtd
