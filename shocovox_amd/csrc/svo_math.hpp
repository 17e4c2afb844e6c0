// Exact single-precision geometry shared by the host octree model, the
// flattener and the gfx950 traversal kernels.
//
// Every function here reproduces the IEEE-754 binary32 operation sequence of
// the reference crate (shocovox-rs 0.11.1) so that host and device produce
// bit-identical trajectories:
//   * no FMA contraction (all sources are built with -ffp-contract=off);
//   * Rust's f32::min / f32::max are NaN-ignoring and, on equal operands,
//     return the receiver (the x86 lowering of llvm.minnum/maxnum:
//     `isnan(a) ? b : (b < a ? b : a)`), spelled out here as selects so the
//     GPU never substitutes v_min_f32 with different signed-zero rules;
//   * f32::signum is +1 for +0.0, -1 for -0.0 and NaN for NaN;
//   * `as` casts from f32 truncate, saturate and map NaN to 0;
//   * conversions V3c<f32> -> V3c<int> use round() (half away from zero);
//   * `x.powf(2.)` is `x * x` (what the optimiser emits for the reference).
// Reference: src/spatial/math/vector.rs:55-81,195-380,
//            src/spatial/raytracing/mod.rs:5-134, src/spatial/mod.rs:31-53,
//            src/spatial/math/mod.rs:11-37, src/spatial/lut.rs:154-253.
#pragma once

#include <cstdint>
#include <cmath>

#if defined(__HIPCC__)
#define SVO_HD __host__ __device__
#else
#define SVO_HD
#endif

namespace svo {

struct V3f {
  float x, y, z;
};

SVO_HD inline V3f v3(float x, float y, float z) { return V3f{x, y, z}; }
SVO_HD inline V3f v3u(float s) { return V3f{s, s, s}; }
SVO_HD inline V3f operator+(V3f a, V3f b) { return V3f{a.x + b.x, a.y + b.y, a.z + b.z}; }
SVO_HD inline V3f operator-(V3f a, V3f b) { return V3f{a.x - b.x, a.y - b.y, a.z - b.z}; }
SVO_HD inline V3f operator*(V3f a, float s) { return V3f{a.x * s, a.y * s, a.z * s}; }
SVO_HD inline V3f operator/(V3f a, float s) { return V3f{a.x / s, a.y / s, a.z / s}; }

// f32::min / f32::max (reference: vector.rs, raytracing/mod.rs:43-44)
SVO_HD inline float rmin(float a, float b) {
  return (a != a) ? b : ((b < a) ? b : a);
}
SVO_HD inline float rmax(float a, float b) {
  return (a != a) ? b : ((b > a) ? b : a);
}

// f32::signum
SVO_HD inline float rsignum(float x) {
  if (x != x) return x;
  return std::signbit(x) ? -1.0f : 1.0f;
}
// rsignum for a non-NaN x (+-1 by the sign bit); +-1 for NaN as well
SVO_HD inline float sign_one(float x) { return copysignf(1.0f, x); }

// `f as i32` (saturating, NaN -> 0)
// Bit (b mod 32) of w.
SVO_HD inline uint32_t bit_of(uint32_t w, uint32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
  // v_bfe_u32 reads the low 5 bits of the offset: one instruction
  return __builtin_amdgcn_ubfe(w, b, 1u);
#else
  return (w >> (b & 31u)) & 1u;
#endif
}

SVO_HD inline int32_t f2i32(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  // v_cvt_i32_f32 truncates toward zero, clamps out-of-range values to
  // [INT32_MIN, INT32_MAX] and converts NaN to 0: Rust's `as i32` in one
  // instruction (the portable form below compiles to compares and branches)
  int32_t r;
  __asm__("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
#endif
  if (x != x) return 0;
  if (x >= 2147483648.0f) return 2147483647;
  if (x < -2147483648.0f) return (-2147483647 - 1);
  return static_cast<int32_t>(x);
}

// `s as i32` for a DDA step component. dda_step returns, per axis, either
// +0.0 or signum(direction), i.e. one of {-1, +1, +0, NaN}; on that domain
// this equals f2i32(s) and f2i32(roundf(s)) (NaN -> 0): one conversion
// instruction on the device, two compares on the host.
SVO_HD inline int32_t step_int(float s) {
#if defined(__HIP_DEVICE_COMPILE__)
  return f2i32(s);
#else
  return s == 1.0f ? 1 : (s == -1.0f ? -1 : 0);
#endif
}

// `f as usize` (saturating, NaN -> 0)
SVO_HD inline uint64_t f2usize(float x) {
  if (!(x > 0.0f)) return 0;  // NaN, zero and negatives
  if (x >= 18446744073709551616.0f) return ~0ull;
  return static_cast<uint64_t>(x);
}

// `f as u32` (saturating, NaN -> 0)
SVO_HD inline uint32_t f2u32(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  // v_cvt_u32_f32: truncation, clamping to [0, UINT32_MAX], NaN -> 0
  uint32_t r;
  __asm__("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
#endif
  if (!(x > 0.0f)) return 0;
  if (x >= 4294967296.0f) return 0xFFFFFFFFu;
  return static_cast<uint32_t>(x);
}

// Correctly rounded quotients and square roots without the compiler's handling
// of extreme exponents (11 instructions a quotient, about 15 a root), for
// operands known to be far from them; the same values, as both are IEEE 754's.
//   * rcp_mid: one Newton step from the hardware's estimate. It rounds
//     correctly for every one of the 2^23 significands. That is a property of
//     gfx950's estimates, held by a test over all of them: from estimates one
//     unit off, 33 significands would round wrong (and 5 in sqrt_mid). Nothing
//     in it depends on the exponent while no operation over- or underflows:
//     |b| in [2^-24, 2^24].
//   * quot_mid(a, b, rcp_mid(b)): Markstein's residual correction (P. Markstein,
//     IBM J. Res. Dev. 34, 1990). It equals a / b for all 2^46 pairs of
//     significands (compared on the device), and the residual is exact for
//     |a| in [2^-60, 2^60]. A +0 numerator over b > 0 gives +0 as well.
//   * sqrt_mid: the same correction from the hardware's reciprocal root, equal
//     to sqrtf for all significands and both exponent parities, for x in
//     [2^-60, 2^100].
// A ray's setup has 12 quotients by 3 divisors and 3 roots, a pixel's direction
// 3 quotients and a root: about 110 of the 1,860 instructions of an 8x8 tile.
#if defined(__HIP_DEVICE_COMPILE__)
__device__ inline float rcp_mid(float b) {
  const float r = __builtin_amdgcn_rcpf(b);
  return fmaf(fmaf(-b, r, 1.0f), r, r);
}
__device__ inline float quot_mid(float a, float b, float rcp_b) {
  const float q = a * rcp_b;
  return fmaf(fmaf(-b, q, a), rcp_b, q);
}
__device__ inline float sqrt_mid(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = x * y;
  return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}
#endif

// V3c<f32>::length: sqrt((x*x + y*y) + z*z)  (vector.rs:75-77)
SVO_HD inline float length(V3f v) {
  const float d2 = (v.x * v.x + v.y * v.y) + v.z * v.z;
#if defined(__HIP_DEVICE_COMPILE__)
  if (d2 >= 0x1p-60f && d2 <= 0x1p60f) return sqrt_mid(d2);
#endif
  return sqrtf(d2);
}
// V3c<f32>::normalized: three divisions by the length (vector.rs:79-81)
SVO_HD inline V3f normalized(V3f v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float d2 = (v.x * v.x + v.y * v.y) + v.z * v.z;
  const float least = fminf(fminf(fabsf(v.x), fabsf(v.y)), fabsf(v.z));
  if (d2 >= 0x1p-40f && d2 <= 0x1p40f && least >= 0x1p-60f) {
    const float len = sqrt_mid(d2);
    const float r = rcp_mid(len);
    return V3f{quot_mid(v.x, len, r), quot_mid(v.y, len, r), quot_mid(v.z, len, r)};
  }
#endif
  return v / length(v);
}

SVO_HD inline V3f cross(V3f a, V3f b) {
  return V3f{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// Octant index of a child region: (x>=h) + 2(z>=h) + 4(y>=h)  (math/mod.rs:11-19)
SVO_HD inline uint32_t hash_region(V3f off, float half) {
  return static_cast<uint32_t>(off.x >= half) + static_cast<uint32_t>(off.z >= half) * 2u +
         static_cast<uint32_t>(off.y >= half) * 4u;
}

// Direction octant: hash_region(1 + dir, 1)  (math/mod.rs:22-26)
SVO_HD inline uint32_t hash_direction(V3f d) { return hash_region(v3u(1.0f) + d, 1.0f); }

constexpr uint32_t OOB_OCTANT = 8;

// OCTANT_OFFSET_REGION_LUT (lut.rs:156-197) as bit triples: x=bit0, y=bit1, z=bit2
SVO_HD inline V3f octant_offset(uint32_t octant) {
  // octant = x + 2z + 4y
  return V3f{static_cast<float>(octant & 1u), static_cast<float>((octant >> 2) & 1u),
             static_cast<float>((octant >> 1) & 1u)};
}

// Mask of the 2x2x2 bitmap cells covered by one octant (lut.rs:199-208)
SVO_HD inline uint64_t octant_bitmap_mask(uint32_t octant) {
  const uint64_t base = 0x0000000000330033ull;
  const uint32_t ox = octant & 1u, oz = (octant >> 1) & 1u, oy = (octant >> 2) & 1u;
  return base << (ox * 2u + oy * 8u + oz * 32u);
}

// The reference's OCTANT_STEP_RESULT_LUT (lut.rs:237-253): the octant reached
// from `octant` after a step with the given component signs, 8 = out of bounds.
SVO_HD inline uint32_t step_octant_signs(uint32_t octant, int sx, int sy, int sz) {
  int x = static_cast<int>(octant & 1u) + sx;
  int y = static_cast<int>((octant >> 2) & 1u) + sy;
  int z = static_cast<int>((octant >> 1) & 1u) + sz;
  if (x < 0 || x > 1 || y < 0 || y > 1 || z < 0 || z > 1) return OOB_OCTANT;
  return static_cast<uint32_t>(x + 2 * z + 4 * y);
}

// step_octant (raytracing/mod.rs:68-80): `(step.c as i32).signum()`
SVO_HD inline uint32_t step_octant(uint32_t octant, V3f step) {
  // step_int is already in {-1, 0, 1}, where signum is the identity
  return step_octant_signs(octant, step_int(step.x), step_int(step.y), step_int(step.z));
}

// Octant bits of three per-axis flags.
SVO_HD inline uint32_t octant_of(bool x, bool y, bool z) {
  return (x ? 1u : 0u) | (z ? 2u : 0u) | (y ? 4u : 0u);
}

// step_octant for a step along the axes of `moved` (octant bits) of a ray
// that runs backwards along the axes of `neg`: an axis steps to the other
// half, or out of the node when the half it is in is already the one the ray
// runs towards (octant bit 1 forwards, 0 backwards).
SVO_HD inline uint32_t step_octant_moved(uint32_t octant, uint32_t moved, uint32_t neg) {
  return ((octant ^ neg) & moved) != 0u ? OOB_OCTANT : octant ^ moved;
}

// Cube{min_position, size}  (spatial/mod.rs:31-53)
struct Cube {
  V3f min;
  float size;
};

// (min + offset * half per axis: the offset is 0 or 1, so the product is
// exact and the fused form rounds the same sum once)
SVO_HD inline Cube child_bounds_for(Cube c, uint32_t octant) {
  const float child_size = c.size / 2.0f;
  const V3f o = octant_offset(octant);
  return Cube{V3f{fmaf(o.x, child_size, c.min.x), fmaf(o.y, child_size, c.min.y),
                  fmaf(o.z, child_size, c.min.z)},
              child_size};
}

// Cube::intersect_ray (raytracing/mod.rs:32-61).
// Returns 0: no intersection, 1: origin inside (impact distance None),
// 2: impact at *t (which may be -0.0).
SVO_HD inline int slabs_hit(float t1, float t2, float t3, float t4, float t5, float t6, float* t) {
  const float tmin = rmax(rmax(rmin(t1, t2), rmin(t3, t4)), rmin(t5, t6));
  const float tmax = rmin(rmin(rmax(t1, t2), rmax(t3, t4)), rmax(t5, t6));
  if (tmax < 0.0f || tmin > tmax) return 0;
  if (tmin < 0.0f) return 1;
  *t = tmin;
  return 2;
}
SVO_HD inline int intersect_ray(Cube c, V3f o, V3f d, float* t) {
  const V3f mx = c.min + v3u(c.size);
  return slabs_hit((c.min.x - o.x) / d.x, (mx.x - o.x) / d.x, (c.min.y - o.y) / d.y,
                   (mx.y - o.y) / d.y, (c.min.z - o.z) / d.z, (mx.z - o.z) / d.z, t);
}

// cube_impact_normal (raytracing/mod.rs:106-134)
SVO_HD inline V3f cube_impact_normal(Cube c, V3f p) {
  const V3f mid = (c.min + v3u(c.size / 2.0f)) - p;
  const float ax = fabsf(mid.x), ay = fabsf(mid.y), az = fabsf(mid.z);
  const float m = rmax(rmax(ax, ay), az);
  const V3f n{ax == m ? -mid.x : 0.0f, ay == m ? -mid.y : 0.0f, az == m ? -mid.z : 0.0f};
#if defined(__HIP_DEVICE_COMPILE__)
  if (m >= 0x1p-20f && m <= 0x1p20f) {  // (the other components are +0)
    const float len = sqrt_mid((n.x * n.x + n.y * n.y) + n.z * n.z);
    const float r = rcp_mid(len);
    return V3f{quot_mid(n.x, len, r), quot_mid(n.y, len, r), quot_mid(n.z, len, r)};
  }
#endif
  return normalized(n);
}

// get_dda_scale_factors (raytracing_on_cpu.rs:99-112)
SVO_HD inline V3f dda_scale_factors(V3f d) {
  const float zx = d.z / d.x, yx = d.y / d.x;
  const float xy = d.x / d.y, zy = d.z / d.y;
  const float xz = d.x / d.z, yz = d.y / d.z;
  return V3f{sqrtf((1.0f + zx * zx) + yx * yx), sqrtf((xy * xy + 1.0f) + zy * zy),
             sqrtf((xz * xz + 1.0f) + yz * yz)};
}

// The two of a ray: intersect_ray(c, o, d, t), and dda_scale_factors(d).
SVO_HD inline int ray_setup(Cube c, V3f o, V3f d, float* t, V3f* scale) {
#if defined(__HIP_DEVICE_COMPILE__)
  const V3f n = c.min - o, x = (c.min + v3u(c.size)) - o;
  const float least = fminf(fminf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
  const float most = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
  const float near = fminf(fminf(fminf(fabsf(n.x), fabsf(n.y)), fabsf(n.z)),
                           fminf(fminf(fabsf(x.x), fabsf(x.y)), fabsf(x.z)));
  const float far = fmaxf(fmaxf(fmaxf(fabsf(n.x), fabsf(n.y)), fabsf(n.z)),
                          fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fabsf(x.z)));
  // (the sum is NaN with any of its operands: the minima and maxima pass over
  // a NaN)
  const bool number = (d.x + d.y) + d.z == (d.x + d.y) + d.z &&
                      (n.x + n.y) + n.z == (n.x + n.y) + n.z;
  if (least >= 0x1p-24f && most <= 0x1p24f && near >= 0x1p-60f && far <= 0x1p60f && number) {
    const float rx = rcp_mid(d.x), ry = rcp_mid(d.y), rz = rcp_mid(d.z);
    const float zx = quot_mid(d.z, d.x, rx), yx = quot_mid(d.y, d.x, rx);
    const float xy = quot_mid(d.x, d.y, ry), zy = quot_mid(d.z, d.y, ry);
    const float xz = quot_mid(d.x, d.z, rz), yz = quot_mid(d.y, d.z, rz);
    *scale = V3f{sqrt_mid((1.0f + zx * zx) + yx * yx), sqrt_mid((xy * xy + 1.0f) + zy * zy),
                 sqrt_mid((xz * xz + 1.0f) + yz * yz)};
    return slabs_hit(quot_mid(n.x, d.x, rx), quot_mid(x.x, d.x, rx), quot_mid(n.y, d.y, ry),
                     quot_mid(x.y, d.y, ry), quot_mid(n.z, d.z, rz), quot_mid(x.z, d.z, rz), t);
  }
#endif
  *scale = dda_scale_factors(d);
  return intersect_ray(c, o, d, t);
}

// c - s * d for a signum s (+1, -1 or NaN): s * d is d negated or not (exact)
// or NaN, so a fused multiply-add, which rounds once, gives exactly the
// reference's product-then-difference (raytracing_on_cpu.rs:136-140).
SVO_HD inline float sub_signed(float c, float s, float d) { return fmaf(-s, d, c); }

// dda_step_to_next_sibling (raytracing_on_cpu.rs:124-152); `sig` is the
// per-ray signum of the direction, hoisted because it never changes.
SVO_HD inline V3f dda_step(V3f dir, V3f sig, V3f* p, Cube b, V3f scale) {
  const V3f diff = *p - b.min;
  const float snx = sub_signed(b.size * rmax(sig.x, 0.0f), sig.x, diff.x);
  const float sny = sub_signed(b.size * rmax(sig.y, 0.0f), sig.y, diff.y);
  const float snz = sub_signed(b.size * rmax(sig.z, 0.0f), sig.z, diff.z);
  const float dx = fabsf(snx * scale.x);
  const float dy = fabsf(sny * scale.y);
  const float dz = fabsf(snz * scale.z);
  // operands are |.| or NaN, where f32::min and fminf (IEEE minNum) agree:
  // NaN yields the other operand and no -0.0 can occur
  const float m = fminf(fminf(dx, dy), dz);
  *p = *p + dir * m;
  return V3f{m == dx ? sig.x : 0.0f, m == dy ? sig.y : 0.0f, m == dz ? sig.z : 0.0f};
}

// dda_step reporting which axes stepped (m == d{x,y,z}, the axes whose step
// component is signum(direction)); the others' components are +0.0.
SVO_HD inline void dda_step_axes(V3f dir, V3f sig, V3f* p, V3f bmin, float size, V3f scale,
                                 bool* ax, bool* ay, bool* az) {
  const V3f diff = *p - bmin;
  const float snx = sub_signed(size * rmax(sig.x, 0.0f), sig.x, diff.x);
  const float sny = sub_signed(size * rmax(sig.y, 0.0f), sig.y, diff.y);
  const float snz = sub_signed(size * rmax(sig.z, 0.0f), sig.z, diff.z);
  const float dx = fabsf(snx * scale.x);
  const float dy = fabsf(sny * scale.y);
  const float dz = fabsf(snz * scale.z);
  const float m = fminf(fminf(dx, dy), dz);
  *p = *p + dir * m;
  *ax = m == dx;
  *ay = m == dy;
  *az = m == dz;
}

// dda_step_axes from the cell's far faces: far = the cell corner the
// direction points to per axis (min + size * max(signum, 0)). The reference's
// size*max(s,0) - s*(p - min) equals far - p on every axis when p - min is
// exact, which holds in the power-of-two layouts (min a multiple of a
// power-of-two size >= 1, coordinates below 2^24, p within about half a
// cell of the cell: min = 0, or Sterbenz's lemma, or p - min in [size, 2 size)
// on the representable grid of size): for s = +1 both are the once-rounded
// real value min + size - p; for s = -1 the reference's is p - min exactly
// and far - p its negation, equal after |.|; for s = NaN every scale factor is
// NaN and both distances are NaN. The reference's distances assume a direction of
// unit length. With another length p leaves the cell by any distance, p - min may
// round, and the two forms part: an impact's last bit for a shorter direction,
// another cell, or none, for some of the rays of a longer one.
// Returns the step length m: when m is not NaN, at least one axis steps
// (fminf returns one of its operands, and m == that operand).
SVO_HD inline float dda_step_far(V3f dir, V3f* p, V3f far, V3f scale, bool* ax, bool* ay,
                                 bool* az) {
  const float dx = fabsf((far.x - p->x) * scale.x);
  const float dy = fabsf((far.y - p->y) * scale.y);
  const float dz = fabsf((far.z - p->z) * scale.z);
  const float m = fminf(fminf(dx, dy), dz);
  *p = *p + dir * m;
  *ax = m == dx;
  *ay = m == dy;
  *az = m == dz;
  return m;
}

// Exact reciprocal of a power of two, 0 for any other value. For s = 2^k the
// products x * 2^-k and the quotient x / 2^k are the same real number, and
// both operations round it once to nearest-even, so `x * pow2_rcp(s)` is
// bit-identical to `x / s` (subnormal results included, as f32 denormals are
// preserved). Reciprocals that would themselves be subnormal are refused.
SVO_HD inline float pow2_rcp(float s) {
  const uint32_t b = __builtin_bit_cast(uint32_t, s);
  const uint32_t e = (b >> 23) & 0xFFu;
  if ((b & 0x807FFFFFu) != 0u || e == 0u || e >= 254u) return 0.0f;
  return __builtin_bit_cast(float, (254u - e) << 23);
}

// x / s, through the exact reciprocal when s is a power of two.
SVO_HD inline float div_by(float x, float s, float rcp) { return rcp != 0.0f ? x * rcp : x / s; }
// div_by for the three components of a vector with one test of the divisor
SVO_HD inline V3f div3_by(V3f v, float s, float rcp) {
  if (rcp != 0.0f) return V3f{v.x * rcp, v.y * rcp, v.z * rcp};
  return V3f{v.x / s, v.y / s, v.z / s};
}

// a - fmodf(a, b) (spatial/math/vector.rs:66-71 as used by the POP at
// raytracing_on_cpu.rs:452-456). For b a power of two >= 1 and 0 < a < 2^24:
// q = floor(a * 2^-k) is exact, q * b is exact, and the reference's
// a - (a - q b) is exactly q b, so floor(a / b) * b is the same value.
// (+-0) - fmodf(+-0, b) is +0.
SVO_HD inline float sub_fmod(float a, float b, float rcp_b) {
  if (a == 0.0f) return 0.0f;
  if (rcp_b != 0.0f && a > 0.0f && a < 16777216.0f && b >= 1.0f) return floorf(a * rcp_b) * b;
  return a - fmodf(a, b);
}

// Palette index value codec (node.rs:354-371)
constexpr uint32_t EMPTY_MARKER = 0xFFFFFFFFu;
constexpr uint32_t NONE16 = 0xFFFFu;
SVO_HD inline uint32_t pix_color_index(uint32_t v) { return v & 0xFFFFu; }
SVO_HD inline uint32_t pix_data_index(uint32_t v) { return (v >> 16) & 0xFFFFu; }

}  // namespace svo
