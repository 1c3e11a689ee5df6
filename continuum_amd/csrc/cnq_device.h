// Device-side geometry of a mask cone for gfx950: vector math, the cone's
// frame and culling tests, and the exact-area accumulation rasterizer.
//
// Semantics follow the reference's GPU kernel,
// crates/continuum-gpu/src/mask_cones.wgsl (cited as "WGSL :line"), with the
// WGSL specification's definitions for normalize (e / length(e)), mix,
// clamp and cross, dot products summed left to right, and no fused
// multiply-adds (the library is built with -ffp-contract=off). Division and
// square root are IEEE correctly rounded (hipcc's default for f32).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cnq {

constexpr uint32_t NONE = 0xffffffffu;
constexpr uint32_t GRID = 8;
constexpr uint32_t BINS = 64;
constexpr float NEAR = 1e-4f;  // WGSL :211
// WGSL's abstract-precision constant 1.0 - 1e-5, rounded once to f32.
constexpr float ONE_MINUS_1EM5 = (float)(1.0 - 1e-5);
// The reference's traversal stack (WGSL :111); a walk deeper than this is
// counted as an overflow.
constexpr uint32_t REF_STACK = 48;

// A branch few waves take: the compiler lays it out of the way and puts what
// it has to spill there.
#define CNQ_RARE(c) __builtin_expect(!!(c), 0)

struct f3 {
  float x, y, z;
};
struct f2 {
  float x, y;
};

__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return f3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return f3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator-(f3 a) { return f3{-a.x, -a.y, -a.z}; }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return f3{a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ f3 operator/(f3 a, float s) { return f3{a.x / s, a.y / s, a.z / s}; }
__device__ __forceinline__ f2 operator+(f2 a, f2 b) { return f2{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ f2 operator-(f2 a, f2 b) { return f2{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ f2 operator*(f2 a, float s) { return f2{a.x * s, a.y * s}; }

__device__ __forceinline__ float dot3(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float dot2(f2 a, f2 b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ f3 cross3(f3 a, f3 b) {
  return f3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float len3(f3 a) { return sqrtf(dot3(a, a)); }
__device__ __forceinline__ f3 norm3(f3 a) { return a / len3(a); }
__device__ __forceinline__ float mn(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float mx(float a, float b) { return b > a ? b : a; }
__device__ __forceinline__ float clampf(float e, float lo, float hi) { return mn(mx(e, lo), hi); }
__device__ __forceinline__ float mixf(float a, float b, float t) { return a * (1.0f - t) + b * t; }
__device__ __forceinline__ f3 ld3(const float* p) { return f3{p[0], p[1], p[2]}; }

// Arctangent after S. L. Moshier's Cephes atanf: reduction by tan(3pi/8) and
// tan(pi/8), then a degree-9 odd minimax polynomial (relative error below
// 2e-7); atan2 by Cephes atan2f's quadrant rule.
constexpr float kPi = 3.14159265358979323846f;
constexpr float kPio2 = 1.57079632679489661923f;
constexpr float kPio4 = 0.78539816339744830962f;

__device__ __forceinline__ float atan_c(float xin) {
  float x = xin;
  float sgn = 1.0f;
  if (x < 0.0f) {
    sgn = -1.0f;
    x = -x;
  }
  float y;
  if (x > 2.414213562373095f) {
    y = kPio2;
    x = -1.0f / x;
  } else if (x > 0.4142135623730950f) {
    y = kPio4;
    x = (x - 1.0f) / (x + 1.0f);
  } else {
    y = 0.0f;
  }
  float z = x * x;
  y = y + ((((8.05374449538e-2f * z - 1.38776856032e-1f) * z + 1.99777106478e-1f) * z - 3.33329491539e-1f) * z *
               x +
           x);
  return sgn * y;
}

__device__ __forceinline__ float atan2_c(float y, float x) {
  if (x == 0.0f) {
    if (y > 0.0f) return kPio2;
    if (y < 0.0f) return -kPio2;
    return 0.0f;
  }
  if (y == 0.0f) return x > 0.0f ? 0.0f : kPi;
  float w = 0.0f;
  if (x < 0.0f) w = y < 0.0f ? -kPi : kPi;
  return w + atan_c(y / x);
}

__device__ __forceinline__ float acos_c(float y) { return atan2_c(sqrtf((1.0f - y) * (1.0f + y)), y); }

// asin(x) = atan2(x, sqrt((1 - x)(1 + x))) for |x| <= 1.
__device__ __forceinline__ float asin_c(float x) { return atan2_c(x, sqrtf((1.0f - x) * (1.0f + x))); }

// Cosine and tangent: S. L. Moshier, Cephes Math Library (sinf.c `cosf`,
// tanf.c): the argument reduced by multiples of pi/4 (pi/4 in three parts),
// then minimax polynomials on [-pi/4, pi/4].
constexpr float kFourOverPi = 1.27323954473516f;
constexpr float kDP1 = 0.78515625f;
constexpr float kDP2 = 2.4187564849853515625e-4f;
constexpr float kDP3 = 3.77489497744594108e-8f;

__device__ __forceinline__ float cos_c(float xin) {
  float x = xin < 0.0f ? -xin : xin;
  int j = (int)(kFourOverPi * x);
  float y = (float)j;
  if (j & 1) {
    j += 1;
    y += 1.0f;
  }
  j &= 7;
  int sign = 1;
  if (j > 3) {
    j -= 4;
    sign = -sign;
  }
  if (j > 1) sign = -sign;
  x = ((x - y * kDP1) - y * kDP2) - y * kDP3;
  const float z = x * x;
  if (j == 1 || j == 2)
    y = ((-1.9515295891e-4f * z + 8.3321608736e-3f) * z - 1.6666654611e-1f) * z * x + x;
  else
    y = ((2.443315711809948e-5f * z - 1.388731625493765e-3f) * z + 4.166664568298827e-2f) * z * z - 0.5f * z + 1.0f;
  return sign < 0 ? -y : y;
}

__device__ __forceinline__ float tan_c(float xin) {
  const float x = xin < 0.0f ? -xin : xin;
  int j = (int)(kFourOverPi * x);
  float y = (float)j;
  if (j & 1) {
    j += 1;
    y += 1.0f;
  }
  const float z = ((x - y * kDP1) - y * kDP2) - y * kDP3;
  const float zz = z * z;
  if (x > 1.0e-4f)
    y = (((((9.38540185543e-3f * zz + 3.11992232697e-3f) * zz + 2.44301354525e-2f) * zz + 5.34112807005e-2f) * zz +
          1.33387994085e-1f) *
             zz +
         3.33331568548e-1f) *
            zz * z +
        z;
  else
    y = z;
  if (j & 2) y = -1.0f / y;
  return xin < 0.0f ? -y : y;
}

// Exponential after Cephes expf: x = n ln2 + r (ln2 in two parts), a
// degree-6 polynomial for e^r, then scaling by 2^n.
__device__ __forceinline__ float exp_c(float x) {
  if (x > 88.72283905206835f) return __builtin_inff();
  if (x < -103.278929903431851103f) return 0.0f;
  float z = floorf(1.44269504088896341f * x + 0.5f);
  x = x - z * 0.693359375f;
  x = x - z * -2.12194440e-4f;
  int n = (int)z;
  float xx = x * x;
  float p = ((((((1.9875691500e-4f * x + 1.3981999507e-3f) * x + 8.3334519073e-3f) * x + 4.1665795894e-2f) * x +
               1.6666665459e-1f) *
                  x +
              5.0000001201e-1f) *
                 xx +
             x) +
            1.0f;
  return ldexpf(p, n);
}

// A mask cone (WGSL :125-146). Light, sky and guard cones take their
// forward axis as the far plane's normal; a lattice cone (a moving rect
// light's, in the view cache) takes the light's plane.
struct Cone {
  f3 apex, right, up, forward;
  float w0, w1, w2, w3;  // window u0, v0, u1, v1
  f3 far_normal;
  float far_offset;
  f3 baxis;  // bounding circular cone: unit axis, cos and sin of the half-angle
  float bcos, bsin;
  // The receiver's horizon (WGSL :147): read only by sky walks (`SKY`),
  // whose cones cull geometry wholly below it; light cones have none.
  f3 horizon;
};

__device__ __forceinline__ f3 direction(const Cone& c, float s, float t) {
  return c.forward + c.right * (c.w0 + s * (c.w2 - c.w0)) + c.up * (c.w1 + t * (c.w3 - c.w1));
}

__device__ __forceinline__ f3 to_local(const Cone& c, f3 p) {
  f3 d = p - c.apex;
  return f3{dot3(c.right, d), dot3(c.up, d), dot3(c.forward, d)};
}

// WGSL :159-168
__device__ __forceinline__ bool in_bound(const Cone& c, f3 p, float r) {
  if (c.bcos < -1.0f) return true;
  f3 d = p - c.apex;
  float len = len3(d);
  if (len <= r) return true;
  float s = r / len;
  float limit = c.bcos * sqrtf(1.0f - s * s) - c.bsin * s;
  return dot3(c.baxis, d) >= limit * len;
}

// WGSL :174-186
__device__ __forceinline__ void bound_cone(Cone& c, f3 axis) {
  float cos_half = 1.0f;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    f3 d = norm3(direction(c, (float)(k & 1u), (float)(k >> 1u)));
    cos_half = mn(cos_half, dot3(axis, d));
  }
  float cos_b = clampf(cos_half - 1e-5f, -1.0f, 1.0f);
  c.baxis = axis;
  c.bcos = cos_b;
  c.bsin = sqrtf(mx(1.0f - cos_b * cos_b, 0.0f));
}

// WGSL :193-201
__device__ __forceinline__ float lambert_edge_unit(f3 n, f3 an, f3 bn) {
  f3 g = cross3(an, bn);
  float len = len3(g);
  if (len > 1e-12f) return atan2_c(len, dot3(an, bn)) * dot3(n, g / len);
  return 0.0f;
}
__device__ __forceinline__ float lambert_edge(f3 n, f3 a, f3 b) { return lambert_edge_unit(n, norm3(a), norm3(b)); }

__device__ __forceinline__ f3 box_corner(f3 lo, f3 hi, uint32_t k) {
  return f3{(k & 1u) ? hi.x : lo.x, (k & 2u) ? hi.y : lo.y, (k & 4u) ? hi.z : lo.z};
}

// A box against a cone (WGSL :159-168 and the culls of :234-255, :519-545),
// settled from the box's centre and half extents: a linear function's
// largest value over the corners is its value at the centre plus |gradient|
// . half extents, about 8 operations a plane where the eight corners take
// 40. The corner tests are f32, so this answers only where its sum clears
// zero by `m`, which bounds the rounding of both sides. Both start from the
// same lo - apex and hi - apex (u = 2^-24): the corner tests' products and
// sums add at most u |d| (4 + 5 |w|); the centre's part 4 u (1 + |w|) |D|; the
// half extents' (their own rounding, the gradient's, its products and sums)
// 6 u (1 + |w|) |H|: in all 11 u (1 + |w|) (|D| + |H|), and m takes 12 u. (The
// tighter the better: a wave goes to the corners when any of its 64 lanes
// has to.) The far plane's test is of world coordinates, so its margin adds
// 8 u (|far offset| + |apex|). A horizon is the caller's normal, of any length:
// its margin is m times its largest component, or m (m alone answered 78 of
// the 3.2 million questions of a test with lengths up to 10^6 wrongly). The
// bounding cone's test of the box's sphere
// (len, r) compares axis . d with cos sqrt(len^2 - r^2) - sin r by
// approximate square roots (1 ulp): with len^2 - r^2 >= 1e-2 len^2 both sides
// are within 4e-6 (|cos| + |sin|) len of `in_bound`'s; the margin allows 2e-5
// of |d|_1 >= len. `in_bound` rounds the centre in world coordinates, up to
// e = u |apex|_1 off: len^2 moves by less than `slip` = 2 s |d|_1 + s^2 with
// s = 13 e, so a box is out of its sphere (which lets everything pass) only
// where len^2 - r^2 exceeds that, and there the two sides move by at most
// 1.02 e len / sqrt(len^2 - r^2) + e <= 11.2 e, of which the margin allows 13.
// (Without `slip` there, 1 to 3 in 10^6 boxes close by an apex 10^5 m from the
// origin are told missed though the sphere holds the apex.) What comes closer
// (or is not a number, or an empty box) goes to the corners (BOX_UNSURE) or to
// `in_bound` (`bound_unsure`: a cone of half a degree leaves most boxes near it
// there, so the planes are asked first).
// With the corners a visit of a triangle hierarchy's node took about 2,000
// cycles (400 instructions), 1,900 of them in the tests; 20,011 scattered
// points by 3 lights went from 7.1 to 5.5 ms, a 1280 x 720 view of the rock
// field from 8.9 to 7.8.
constexpr uint32_t BOX_OUT = 0, BOX_CROSS = 1, BOX_INSIDE = 2, BOX_UNSURE = 3;

__device__ __forceinline__ float fdot3(f3 a, f3 b) {  // fused: for bounds only
  return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.y, b.y, a.x * b.x));
}
__device__ __forceinline__ f3 abs3(f3 a) { return f3{fabsf(a.x), fabsf(a.y), fabsf(a.z)}; }
__device__ __forceinline__ float sum3(f3 a) { return a.x + a.y + a.z; }

// A cone's part of the tests: the far plane seen from the apex and its
// margin, the window's factor, the bounding cone's margins, the horizon's
// factor (sky walks).
struct ConeMargins {
  float far, far_margin, window, bound, bound_apex, horizon;
};
__device__ __forceinline__ ConeMargins cone_margins(const Cone& c) {
  const float apex = sum3(abs3(c.apex));
  return ConeMargins{c.far_offset - fdot3(c.far_normal, c.apex), 4.8e-7f * (fabsf(c.far_offset) + apex),
                     1.0f + fmaxf(fmaxf(fabsf(c.w0), fabsf(c.w1)), fmaxf(fabsf(c.w2), fabsf(c.w3))),
                     2e-5f * (fabsf(c.bcos) + fabsf(c.bsin)), 7.8e-7f * apex,
                     fmaxf(fmaxf(1.0f, fabsf(c.horizon.x)), fmaxf(fabsf(c.horizon.y), fabsf(c.horizon.z)))};
}

// The box in the cone's frame: its centre there, half extents (world) and m.
struct BoxQuick {
  f3 half, local;
  float m;
  bool bound_unsure;
};

// BOX_OUT, BOX_CROSS (in every plane's reach, but a corner lies before the
// near or past the far plane), BOX_INSIDE (every corner between them) or
// BOX_UNSURE. Without INSIDE the last two planes' inner sides are not asked
// for, and BOX_CROSS means "not out".
template <bool SKY, bool INSIDE>
__device__ __forceinline__ uint32_t box_quick(const Cone& c, const ConeMargins& cm, f3 lo, f3 hi, BoxQuick& b) {
  const f3 dlo = lo - c.apex, dhi = hi - c.apex;
  const f3 d = (dlo + dhi) * 0.5f;
  b.half = abs3((dhi - dlo) * 0.5f);
  const float d1 = sum3(abs3(d));
  b.m = __builtin_fmaf(7.2e-7f, d1 + sum3(b.half), 1e-30f);
  // The bounding cone first: often it settles every lane a node was left for.
  const float l2 = fdot3(d, d), r2 = fdot3(b.half, b.half), t = l2 - r2;
  const float rhs = __builtin_fmaf(c.bcos, __builtin_amdgcn_sqrtf(fmaxf(t, 0.0f)),
                                   -(c.bsin * __builtin_amdgcn_sqrtf(r2)));
  const float over = fdot3(c.baxis, d) - rhs, bm = __builtin_fmaf(cm.bound, d1, cm.bound_apex);
  const float slip = cm.bound_apex * __builtin_fmaf(2.0f, d1, cm.bound_apex);
  const bool sized = (t > __builtin_fmaf(1e-2f, l2, slip)) & (l2 > 1e-20f) & (l2 < 1e30f);
  if (sized & (over < -bm)) return BOX_OUT;
  b.local = f3{fdot3(c.right, d), fdot3(c.up, d), fdot3(c.forward, d)};
  // The least of the four window planes' largest values.
  auto reach = [&](f3 axis, float w) {  // |axis - w forward| . half
    asm volatile("" : "+v"(w));  // (twelve products, not twelve registers for the whole walk)
    const f3 n{__builtin_fmaf(-w, c.forward.x, axis.x), __builtin_fmaf(-w, c.forward.y, axis.y),
               __builtin_fmaf(-w, c.forward.z, axis.z)};
    return fdot3(abs3(n), b.half);
  };
  const float side = fminf(
      fminf(__builtin_fmaf(-c.w0, b.local.z, b.local.x) + reach(c.right, c.w0),
            __builtin_fmaf(c.w2, b.local.z, -b.local.x) + reach(c.right, c.w2)),
      fminf(__builtin_fmaf(-c.w1, b.local.z, b.local.y) + reach(c.up, c.w1),
            __builtin_fmaf(c.w3, b.local.z, -b.local.y) + reach(c.up, c.w3)));
  const float mw = b.m * cm.window;
  const float ez = fdot3(abs3(c.forward), b.half);
  const float fc = cm.far - fdot3(c.far_normal, d), fe = fdot3(abs3(c.far_normal), b.half);
  const float mf = b.m + cm.far_margin;
  const float zr = b.local.z + ez - NEAR, fr = fc + fe;
  bool out = (side < -mw) | (zr < -b.m) | (fr < -mf);
  bool sure = (side > mw) & (zr > b.m) & (fr > mf);
  b.bound_unsure = !((sized & (over > bm)) |
                     ((l2 + slip < 0.9999f * r2) & (r2 > 1e-20f) & (r2 < 1e30f)) |
                     (c.bcos < -1.0f));
  if (SKY) {
    // (a zero horizon culls nothing)
    const float hr = fdot3(c.horizon, d) + fdot3(abs3(c.horizon), b.half);
    const float mh = b.m * cm.horizon;
    out = out | (hr < -mh);
    sure = sure & ((hr > mh) | ((c.horizon.x == 0.0f) & (c.horizon.y == 0.0f) & (c.horizon.z == 0.0f)));
  }
  uint32_t r = BOX_CROSS;
  if (INSIDE) {
    const float zi = b.local.z - ez - NEAR, fi = fc - fe;
    const bool in = (zi > b.m) & (fi > mf);
    sure = sure & (in | (zi < -b.m) | (fi < -mf));
    r = in ? BOX_INSIDE : BOX_CROSS;
  }
  return out ? BOX_OUT : (sure ? r : BOX_UNSURE);
}

// The planes' part from the eight corners (never BOX_UNSURE).
template <bool SKY>
__device__ __forceinline__ uint32_t box_corners(const Cone& c, f3 lo, f3 hi) {
  bool far_out = true, near_out = true, out_u0 = true, out_u1 = true, out_v0 = true, out_v1 = true;
  bool below = SKY, inside = true;
#pragma unroll 1
  for (uint32_t k = 0; k < 8; k++) {
    f3 corner = box_corner(lo, hi, k);
    if (SKY && dot3(c.horizon, corner - c.apex) >= 0.0f) below = false;
    if (c.far_offset - dot3(c.far_normal, corner) >= 0.0f)
      far_out = false;
    else
      inside = false;
    f3 p = to_local(c, corner);
    if (p.z >= NEAR)
      near_out = false;
    else
      inside = false;
    if (p.x - c.w0 * p.z >= 0.0f) out_u0 = false;
    if (c.w2 * p.z - p.x >= 0.0f) out_u1 = false;
    if (p.y - c.w1 * p.z >= 0.0f) out_v0 = false;
    if (c.w3 * p.z - p.y >= 0.0f) out_v1 = false;
  }
  if (far_out || near_out || out_u0 || out_u1 || out_v0 || out_v1 || below) return BOX_OUT;
  return inside ? BOX_INSIDE : BOX_CROSS;
}

// WGSL :234-255; the horizon test only with SKY (light cones have none)
template <bool SKY = false>
__device__ __forceinline__ bool may_touch_box(const Cone& c, const ConeMargins& cm, f3 lo, f3 hi) {
  BoxQuick b;
  uint32_t side = box_quick<SKY, false>(c, cm, lo, hi, b);
  if (side == BOX_UNSURE) side = box_corners<SKY>(c, lo, hi);
  if (side == BOX_OUT) return false;
  return !b.bound_unsure || in_bound(c, (lo + hi) * 0.5f, 0.5f * len3(hi - lo));
}

// WGSL :213-232 (the horizon test only with SKY)
template <bool SKY = false>
__device__ __forceinline__ bool may_touch(const Cone& c, f3 v0, f3 v1, f3 v2) {
  float f0 = c.far_offset - dot3(c.far_normal, v0);
  float f1 = c.far_offset - dot3(c.far_normal, v1);
  float f2 = c.far_offset - dot3(c.far_normal, v2);
  if (f0 < 0.0f && f1 < 0.0f && f2 < 0.0f) return false;
  if (SKY && dot3(c.horizon, v0 - c.apex) < 0.0f && dot3(c.horizon, v1 - c.apex) < 0.0f &&
      dot3(c.horizon, v2 - c.apex) < 0.0f)
    return false;
  f3 p0 = to_local(c, v0), p1 = to_local(c, v1), p2 = to_local(c, v2);
  if (p0.z < NEAR && p1.z < NEAR && p2.z < NEAR) return false;
  if (p0.x - c.w0 * p0.z < 0.0f && p1.x - c.w0 * p1.z < 0.0f && p2.x - c.w0 * p2.z < 0.0f) return false;
  if (c.w2 * p0.z - p0.x < 0.0f && c.w2 * p1.z - p1.x < 0.0f && c.w2 * p2.z - p2.x < 0.0f) return false;
  if (p0.y - c.w1 * p0.z < 0.0f && p1.y - c.w1 * p1.z < 0.0f && p2.y - c.w1 * p2.z < 0.0f) return false;
  if (c.w3 * p0.z - p0.y < 0.0f && c.w3 * p1.z - p1.y < 0.0f && c.w3 * p2.z - p2.y < 0.0f) return false;
  return true;
}

// ---- Per-query working memory, in LDS and lane-interleaved (cell s of lane
// l at s * 64 + l), so every access is bank-conflict free whatever cell each
// lane touches: the 66-cell accumulation buffer (a row's last cell spills
// into the next row's first two), then the polygon a draw works on, 7
// vertices of 2 cells. 80 cells are 20,480 B a wave, an eighth of a CU's
// 160 KB: two waves a SIMD.
constexpr uint32_t ACC_CELLS = 66;
constexpr uint32_t GRID_VERTS = 7;  // a window's square cut by a triangle's three edges
constexpr uint32_t GRID_POLY = ACC_CELLS;
constexpr uint32_t WALK_CELLS = ACC_CELLS + 2 * GRID_VERTS;
// The rare general clips (a triangle crossing the near or the far plane, a
// polygon outgrowing the 7 vertices, horizon-clipped quads of the weights)
// work in 70 slots: a 3D polygon of up to 10 vertices at slots 0-29, its
// clip target at 30-59; 2D polygons at 30-49 and 50-69 once the 3D clip is
// done. They lie in the lane's private memory (scratch, stride 1); the cone
// kernel's one-wave variant keeps them in LDS too (stride 64).
constexpr uint32_t POLY_SLOTS = 70;
constexpr uint32_t POLY_STRIDE = 1;
constexpr uint32_t POLY_STRIDE_LDS = 64;
// Waves per SIMD the walk kernels are compiled for (their registers are
// limited to 256 a lane; the LDS, 20 KB a wave, allows it).
constexpr int WALK_WAVES = 2;
constexpr uint32_t P3A = 0, P3B = 30, Q2A = 30, Q2B = 50;
constexpr uint32_t MAX_POLY = 10;  // WGSL :11

struct Lane {
  float* acc;       // this lane's accumulation cell 0
  float* poly;      // this lane's polygon slot 0
  uint32_t pstride;  // polygon slot i at poly[i * pstride]
  uint32_t span_lo, span_hi;
  // The accumulator is in LDS: an LDS atomic add (ds_add_f32) needs no read
  // round trip, and rounds as v_add_f32 does (round to nearest even,
  // denormals kept: checked bit for bit on the device). A lane's adds to its
  // own cells take effect in program order, so each cell sums its terms in
  // the same order as the plain read-add-write.
  __device__ __forceinline__ void add(uint32_t cell, float v) {
    __hip_atomic_fetch_add((__attribute__((address_space(3))) float*)(acc + cell * 64u), v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ float get(uint32_t cell) const { return acc[cell * 64u]; }
  __device__ __forceinline__ void set(uint32_t cell, float v) { acc[cell * 64u] = v; }
  // Vertex i of the draw's polygon.
  __device__ __forceinline__ f2 vert(uint32_t i) const {
    const float* p = acc + (GRID_POLY + 2u * i) * 64u;
    return f2{p[0], p[64]};
  }
  __device__ __forceinline__ void put_vert(uint32_t i, f2 v) {
    float* p = acc + (GRID_POLY + 2u * i) * 64u;
    p[0] = v.x;
    p[64] = v.y;
  }
  __device__ __forceinline__ f3 p3(uint32_t base, uint32_t i) const {
    const float* p = poly + (base + 3u * i) * pstride;
    return f3{p[0], p[pstride], p[2 * pstride]};
  }
  __device__ __forceinline__ void put3(uint32_t base, uint32_t i, f3 v) {
    float* p = poly + (base + 3u * i) * pstride;
    p[0] = v.x;
    p[pstride] = v.y;
    p[2 * pstride] = v.z;
  }
  __device__ __forceinline__ f2 p2(uint32_t base, uint32_t i) const {
    const float* p = poly + (base + 2u * i) * pstride;
    return f2{p[0], p[pstride]};
  }
  __device__ __forceinline__ void put2(uint32_t base, uint32_t i, f2 v) {
    float* p = poly + (base + 2u * i) * pstride;
    p[0] = v.x;
    p[pstride] = v.y;
  }
};

// WGSL :297-348
__device__ __forceinline__ void draw_edge(Lane& acc, f2 q0, f2 q1, float weight) {
  if (fabsf(q0.y - q1.y) <= 1.1920929e-7f) return;
  float dir = 1.0f;
  f2 p0 = q0, p1 = q1;
  if (q0.y > q1.y) {
    dir = -1.0f;
    p0 = q1;
    p1 = q0;
  }
  float dxdy = (p1.x - p0.x) / (p1.y - p0.y);
  float x = p0.x;
  uint32_t yc = (uint32_t)ceilf(p1.y);
  uint32_t y_end = yc < GRID ? yc : GRID;
  const uint32_t y_begin = (uint32_t)p0.y;
  // The rows' span, once per edge (the rows run upward), and the signed
  // weight: dir is +-1, so (dy dir) w and dy (dir w) are the same float.
  if (y_begin < y_end) {
    acc.span_lo = acc.span_lo < y_begin * GRID ? acc.span_lo : y_begin * GRID;
    const uint32_t hi = (y_end - 1u) * GRID + GRID + 1u;
    acc.span_hi = acc.span_hi > hi ? acc.span_hi : hi;
  }
  const float dir_weight = dir * weight;
  for (uint32_t y = y_begin; y < y_end; y++) {
    uint32_t row = y * GRID;
    float dy = mn((float)(y + 1u), p1.y) - mx((float)y, p0.y);
    float x_next = clampf(x + dxdy * dy, 0.0f, (float)GRID);
    float d = dy * dir_weight;
    float x0 = mn(x, x_next);
    float x1 = mx(x, x_next);
    float x0_floor = floorf(x0);
    uint32_t x0i = (uint32_t)x0_floor;
    float x1_ceil = ceilf(x1);
    uint32_t x1i = (uint32_t)x1_ceil;
    if (x1i <= x0i + 1u) {
      float xmf = 0.5f * (x + x_next) - x0_floor;
      acc.add(row + x0i, d - d * xmf);
      acc.add(row + x0i + 1u, d * xmf);
    } else {
      float s = 1.0f / (x1 - x0);
      float x0f = x0 - x0_floor;
      float a0 = 0.5f * s * (1.0f - x0f) * (1.0f - x0f);
      float x1f = x1 - x1_ceil + 1.0f;
      float am = 0.5f * s * x1f * x1f;
      acc.add(row + x0i, d * a0);
      if (x1i == x0i + 2u) {
        acc.add(row + x0i + 1u, d * (1.0f - a0 - am));
      } else {
        float a1 = s * (1.5f - x0f);
        acc.add(row + x0i + 1u, d * (a1 - a0));
        for (uint32_t xi = x0i + 2u; xi < x1i - 1u; xi++) acc.add(row + xi, d * s);
        float a2 = a1 + (float)(x1i - x0i - 3u) * s;
        acc.add(row + x1i - 1u, d * (1.0f - a2 - am));
      }
      acc.add(row + x1i, d * am);
    }
    x = x_next;
  }
}

__device__ __forceinline__ f2 clamp_grid(f2 v) {
  const float g = (float)GRID;
  return f2{clampf(v.x, 0.0f, g), clampf(v.y, 0.0f, g)};
}

// WGSL :264-278: keeps dot(normal, x) <= offset; crossings from the kept end.
// Polygon `src` (n vertices) to `dst`; returns the new count (at most 10).
__device__ __forceinline__ uint32_t clip_plane3(Lane& L, uint32_t src, uint32_t n, f3 normal, float offset,
                                                uint32_t dst) {
  uint32_t m = 0;
  if (n == 0) return 0;
  // The source's vertices in one batch of loads (slots past n re-read vertex 0).
  f3 v[MAX_POLY];
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++) v[i] = L.p3(src, i < n ? i : 0u);
  const f3 first = v[0];
  f3 a = first;
  float da = offset - dot3(normal, a);
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++) {
    if (i < n) {
      const f3 b = i + 1 < n ? v[i + 1 < MAX_POLY ? i + 1 : 0] : first;
      const float db = offset - dot3(normal, b);
      if (da >= 0.0f && m < MAX_POLY) L.put3(dst, m++, a);
      if (da >= 0.0f && db < 0.0f && m < MAX_POLY) L.put3(dst, m++, a + (b - a) * (da / (da - db)));
      if (da < 0.0f && db >= 0.0f && m < MAX_POLY) L.put3(dst, m++, b + (a - b) * (db / (db - da)));
      a = b;
      da = db;
    }
  }
  return m;
}

// WGSL :280-294, in the projected plane. The source polygon's vertices are
// read in one batch of loads before the clip (slots past `n` re-read vertex
// 0 and go unused), so a pass waits on memory once, not once per vertex;
// the arithmetic and the order of the outputs are the loop's own.
__device__ __forceinline__ uint32_t clip_line2(Lane& L, uint32_t src, uint32_t n, f2 normal, float offset,
                                               uint32_t dst) {
  uint32_t m = 0;
  if (n == 0) return 0;
  f2 v[MAX_POLY];
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++) v[i] = L.p2(src, i < n ? i : 0u);
  const f2 first = v[0];
  f2 a = first;
  float da = offset - dot2(normal, a);
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++) {
    if (i < n) {
      const f2 b = i + 1 < n ? v[i + 1 < MAX_POLY ? i + 1 : 0] : first;
      const float db = offset - dot2(normal, b);
      if (da >= 0.0f && m < MAX_POLY) L.put2(dst, m++, a);
      if (da >= 0.0f && db < 0.0f && m < MAX_POLY) L.put2(dst, m++, a + (b - a) * (da / (da - db)));
      if (da < 0.0f && db >= 0.0f && m < MAX_POLY) L.put2(dst, m++, b + (a - b) * (db / (db - da)));
      a = b;
      da = db;
    }
  }
  return m;
}

// The four clips to [0, 8]^2 (WGSL :432-437: x >= 0, x <= 8, y >= 0, y <= 8,
// in that order), ping-ponging between the two 2D slots; `at` is where the
// polygon is, and is where it ends up.
__device__ __forceinline__ uint32_t clip_to_grid(Lane& L, uint32_t& at, uint32_t n) {
  const float g = (float)GRID;
  const uint32_t other = at == Q2A ? Q2B : Q2A;
#pragma unroll 1
  for (uint32_t k = 0; k < 4; k++) {
    const f2 normal{k == 0 ? -1.0f : (k == 1 ? 1.0f : 0.0f), k == 2 ? -1.0f : (k == 3 ? 1.0f : 0.0f)};
    const bool odd = (k & 1u) != 0;
    n = clip_line2(L, odd ? other : at, n, normal, odd ? g : 0.0f, odd ? at : other);
  }
  return n;
}

// Draws the edges of the polygon in LDS (n <= 8 vertices, the eighth in
// `last`), in order; each next vertex is read while an edge is drawn.
__device__ __forceinline__ void draw_poly(Lane& L, uint32_t n, f2 last, float weight) {
  const f2 first = L.vert(0);
  f2 a = first, b = L.vert(1);
  for (uint32_t i = 1; i <= n; i++) {
    const f2 ahead = i + 1u < GRID_VERTS ? L.vert(i + 1u) : last;
    const f2 to = i < n ? b : first;
    draw_edge(L, a, to, weight);
    a = to;
    b = ahead;
  }
}

// A polygon the general clips left in private memory, brought to LDS; with
// nine or ten vertices it is drawn from where it is instead (true).
__device__ __forceinline__ bool draw_general(Lane& L, uint32_t at, uint32_t n, f2& last, float weight) {
  if (CNQ_RARE(n > GRID_VERTS + 1u)) {
    const f2 first = clamp_grid(L.p2(at, 0));
    f2 a = first;
#pragma unroll 1
    for (uint32_t i = 1; i <= n; i++) {
      const f2 b = i < n ? clamp_grid(L.p2(at, i)) : first;
      draw_edge(L, a, b, weight);
      a = b;
    }
    return true;
  }
#pragma unroll 1
  for (uint32_t i = 0; i < n && i < GRID_VERTS; i++) L.put_vert(i, clamp_grid(L.p2(at, i)));
  if (n > GRID_VERTS) last = clamp_grid(L.p2(at, GRID_VERTS));
  return false;
}

// `clip_line2` of the polygon in LDS, in place: at most N (<= 7) vertices
// in, `bad` (and nothing changed) when it would leave more than 7 or when
// the line crosses more than one edge each way, as only rounding can make
// it. A convex polygon loses one run of vertices for the two crossings, so
// the distances give a mask of kept vertices, its edges the crossings'
// places, and only the two crossings are computed (the loop over ten vertices
// computes one for every vertex some lane crosses at); the vertices after the
// lost run move to their new places. Arithmetic and order are clip_line2's.
template <uint32_t N>
__device__ __forceinline__ uint32_t clip_line_lds(Lane& L, uint32_t n, f2 normal, float offset, bool& bad,
                                                  bool& out_of_grid) {
  f2 v[N];
#pragma unroll
  for (uint32_t k = 0; k < N; k++) v[k] = L.vert(k);
  uint32_t in = 0;
#pragma unroll
  for (uint32_t k = 0; k < N; k++) in |= offset - dot2(normal, v[k]) >= 0.0f ? 1u << k : 0u;
  const uint32_t full = (1u << n) - 1u;
  in &= full;
  if (in == full || n == 0) return n;
  if (in == 0) return 0;
  const uint32_t next = (in >> 1) | ((in & 1u) << (n - 1u));
  const uint32_t leave = in & ~next, enter = ~in & next;
  const uint32_t i = (uint32_t)__builtin_ctz(leave), j = (uint32_t)__builtin_ctz(enter);
  const bool kept0 = (in & 1u) != 0;
  const uint32_t m = kept0 ? n + i + 2u - j : i + 2u - j;
  if (CNQ_RARE((leave & (leave - 1u)) != 0 || m > GRID_VERTS)) {
    bad = true;
    return n;
  }
  const f2 a = L.vert(i), b = L.vert(i + 1u == n ? 0u : i + 1u);
  const f2 c = L.vert(j), d = L.vert(j + 1u == n ? 0u : j + 1u);
  const float da = offset - dot2(normal, a), db = offset - dot2(normal, b);
  const float dc = offset - dot2(normal, c), dd = offset - dot2(normal, d);
  const f2 x = a + (b - a) * (da / (da - db));
  const f2 y = d + (c - d) * (dd / (dd - dc));
  // Vertex 0 kept: v0..vi, x, y, v(j+1)..; lost: y, v(j+1)..vi, x.
  const uint32_t shift = kept0 ? i + 2u - j : 0u - j;
#pragma unroll
  for (uint32_t k = 1; k < N; k++)
    if (k > j && k < n) L.put_vert(k + shift, v[k]);
  L.put_vert(kept0 ? i + 1u : i - j + 1u, x);
  L.put_vert(kept0 ? i + 2u : 0u, y);
  const float g = (float)GRID;
  out_of_grid = out_of_grid || x.x < 0.0f || x.y < 0.0f || x.x > g || x.y > g || y.x < 0.0f || y.y < 0.0f ||
                y.x > g || y.y > g;
  return m;
}

__device__ __forceinline__ bool in_window(const Cone& c, f3 v) {
  return !(v.x < c.w0 * v.z || v.x > c.w2 * v.z || v.y < c.w1 * v.z || v.y > c.w3 * v.z);
}

__device__ __forceinline__ f2 project(const Cone& c, f3 v, float su, float sv) {
  return f2{(v.x / v.z - c.w0) * su, (v.y / v.z - c.w1) * sv};
}

__device__ __forceinline__ bool in_grid(f2 q) {
  const float g = (float)GRID;
  return !(q.x < 0.0f || q.y < 0.0f || q.x > g || q.y > g);
}

// The general path of `rasterize` (WGSL :358-431) up to the grid clip: the
// triangle as a polygon, clipped by the far plane (`far_clip`) and the near
// plane where it crosses them, then either projected (wholly in the window)
// or the window's square clipped by the planes through the apex and each of
// its edges. Leaves the 2D polygon at `at` and returns its vertex count (0:
// nothing to draw); `grid_clip`: a vertex lies outside the grid. Without a
// far clip the caller passes the triangle's local corners (l0, l1, l2); where
// all three lie in front of the near plane (the common case) the edge planes
// come from them in registers, and the 3D polygon never goes to memory.
__device__ __forceinline__ uint32_t general_polygon(const Cone& c, Lane& L, f3 v0, f3 v1, f3 v2, bool far_clip,
                                                    f3 l0, f3 l1, f3 l2, float su, float sv, uint32_t& at,
                                                    bool& grid_clip) {
  const float g = (float)GRID;
  grid_clip = false;
  at = Q2A;
  uint32_t n = 3;
  bool all_near_ok = true, all_in_window = true, in_regs = false;
  if (!far_clip) {
    all_near_ok = l0.z >= NEAR && l1.z >= NEAR && l2.z >= NEAR;
    all_in_window = in_window(c, l0) && in_window(c, l1) && in_window(c, l2);
    in_regs = all_near_ok;
    if (!all_near_ok) {
      L.put3(P3A, 0, l0);
      L.put3(P3A, 1, l1);
      L.put3(P3A, 2, l2);
    }
  } else {
    L.put3(P3A, 0, v0);
    L.put3(P3A, 1, v1);
    L.put3(P3A, 2, v2);
    n = clip_plane3(L, P3A, n, c.far_normal, c.far_offset, P3B);
    for (uint32_t i = 0; i < n; i++) {
      const f3 v = to_local(c, L.p3(P3B, i));
      L.put3(P3A, i, v);
      if (v.z < NEAR) all_near_ok = false;
      if (!in_window(c, v)) all_in_window = false;
    }
  }
  if (!all_near_ok) {
    n = clip_plane3(L, P3A, n, f3{0.0f, 0.0f, -1.0f}, -NEAR, P3B);
    for (uint32_t i = 0; i < n; i++) L.put3(P3A, i, L.p3(P3B, i));
  }
  if (n < 3) return 0;
  uint32_t qn;
  if (all_near_ok && all_in_window) {
    qn = n;
    for (uint32_t i = 0; i < n; i++) {
      const f3 p = in_regs ? (i == 0 ? l0 : (i == 1 ? l1 : l2)) : L.p3(P3A, i);
      L.put2(Q2A, i, project(c, p, su, sv));
    }
  } else {
    // The window's square clipped by the planes through the apex and each
    // edge, with the whole triangle's winding (WGSL :376-425).
    const f3 t0 = far_clip ? to_local(c, v0) : l0, t1 = far_clip ? to_local(c, v1) : l1,
             t2 = far_clip ? to_local(c, v2) : l2;
    const float d = dot3(t0, cross3(t1, t2));
    if (d == 0.0f) return 0;
    const float side = d > 0.0f ? 1.0f : -1.0f;
    qn = 4;
    L.put2(Q2A, 0, f2{0.0f, 0.0f});
    L.put2(Q2A, 2, f2{g, g});
    if (side > 0.0f) {
      L.put2(Q2A, 1, f2{g, 0.0f});
      L.put2(Q2A, 3, f2{0.0f, g});
    } else {
      L.put2(Q2A, 1, f2{0.0f, g});
      L.put2(Q2A, 3, f2{g, 0.0f});
    }
    for (uint32_t i = 0; i < n; i++) {
      f3 p, q;
      if (in_regs) {
        p = i == 0 ? l0 : (i == 1 ? l1 : l2);
        q = i == 0 ? l1 : (i == 1 ? l2 : l0);
      } else {
        p = L.p3(P3A, i);
        q = L.p3(P3A, i + 1 == n ? 0 : i + 1);
      }
      const f3 e = cross3(p, q);
      const float len = len3(e);
      if (len == 0.0f) continue;
      const f3 k = e * (side / len);
      const uint32_t to = at == Q2A ? Q2B : Q2A;
      qn = clip_line2(L, at, qn, f2{-k.x / su, -k.y / sv}, k.x * c.w0 + k.y * c.w1 + k.z, to);
      at = to;
    }
  }
  f2 v[MAX_POLY];
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++) v[i] = L.p2(at, i < qn ? i : 0u);
#pragma unroll
  for (uint32_t i = 0; i < MAX_POLY; i++)
    if (i < qn && !in_grid(v[i])) grid_clip = true;
  return qn;
}

// The window's square in LDS, cut by the planes through the apex and each
// edge of a triangle in front of the near plane (local corners l0..l2), with
// the triangle's winding (WGSL :376-425). Returns the vertices left; `bad`
// when general_polygon has to build it instead.
__device__ __forceinline__ uint32_t window_polygon(const Cone& c, Lane& L, f3 l0, f3 l1, f3 l2, float su, float sv,
                                                   bool& bad) {
  const float g = (float)GRID;
  const float d = dot3(l0, cross3(l1, l2));
  if (d == 0.0f) return 0;
  const bool ccw = d > 0.0f;
  const float side = ccw ? 1.0f : -1.0f;
  L.put_vert(0, f2{0.0f, 0.0f});
  L.put_vert(1, ccw ? f2{g, 0.0f} : f2{0.0f, g});
  L.put_vert(2, f2{g, g});
  L.put_vert(3, ccw ? f2{0.0f, g} : f2{g, 0.0f});
  uint32_t n = 4;
  bool outside = false;
#pragma unroll 1
  for (uint32_t i = 0; i < 3; i++) {
    const f3 p = i == 0 ? l0 : (i == 1 ? l1 : l2), q = i == 0 ? l1 : (i == 1 ? l2 : l0);
    const f3 e = cross3(p, q);
    const float len = len3(e);
    if (len == 0.0f) continue;
    const f3 k = e * (side / len);
    const f2 normal{-k.x / su, -k.y / sv};
    const float offset = k.x * c.w0 + k.y * c.w1 + k.z;
    if (!(fabsf(normal.x) < 1e30f && fabsf(normal.y) < 1e30f && fabsf(offset) < 1e30f)) bad = true;
    if (!bad) n = clip_line_lds<6>(L, n, normal, offset, bad, outside);
  }
  bad = bad || outside;
  return n;
}

// WGSL :350-451. A triangle in front of the near plane and before the far
// plane becomes a polygon of at most 7 vertices in LDS: itself projected
// when it lies in the window, else the window's square cut by its edges. The
// rest (a plane crossed, rounding that left the grid) is built by the general
// clips in private memory and, up to eight vertices of it, brought to LDS (the
// eighth in registers; nine or ten are drawn from where they are). One loop
// then draws whatever the lanes hold. (The general clips used to take
// every triangle that crosses the window: 8,900 cycles a round of draws on
// the courtyard, most of them round trips to private memory and crossings
// computed at every vertex, and 3,500 more where lanes drew whole triangles
// beside them.)
__device__ __forceinline__ bool rasterize(const Cone& c, Lane& L, f3 v0, f3 v1, f3 v2, float weight) {
  const float f0 = c.far_offset - dot3(c.far_normal, v0);
  const float f1 = c.far_offset - dot3(c.far_normal, v1);
  const float f2_ = c.far_offset - dot3(c.far_normal, v2);
  const bool far_clip = f0 < 0.0f || f1 < 0.0f || f2_ < 0.0f;
  const float su = (float)GRID / (c.w2 - c.w0);
  const float sv = (float)GRID / (c.w3 - c.w1);
  const f3 l0 = to_local(c, v0), l1 = to_local(c, v1), l2 = to_local(c, v2);
  uint32_t n = 0;
  bool general = far_clip || !(l0.z >= NEAR && l1.z >= NEAR && l2.z >= NEAR);
  if (!general) {
    if (in_window(c, l0) && in_window(c, l1) && in_window(c, l2)) {
      const f2 q0 = project(c, l0, su, sv), q1 = project(c, l1, su, sv), q2 = project(c, l2, su, sv);
      L.put_vert(0, q0);
      L.put_vert(1, q1);
      L.put_vert(2, q2);
      n = 3;
      // (rounding can put a corner a hair outside the grid)
      general = !(in_grid(q0) && in_grid(q1) && in_grid(q2));
    } else {
      n = window_polygon(c, L, l0, l1, l2, su, sv, general);
    }
  }
  f2 last{0.0f, 0.0f};
  if (CNQ_RARE(general)) {
    uint32_t at = Q2A;
    bool grid_clip = false;
    n = general_polygon(c, L, v0, v1, v2, far_clip, l0, l1, l2, su, sv, at, grid_clip);
    if (grid_clip) n = clip_to_grid(L, at, n);
    if (draw_general(L, at, n, last, weight)) return true;
  }
  if (n < 3) return false;
  draw_poly(L, n, last, weight);
  return true;
}

}  // namespace cnq
