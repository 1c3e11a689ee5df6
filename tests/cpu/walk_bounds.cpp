// The walk's short cuts against the plain tests they stand for, on the CPU:
// the device headers compiled for one lane (no contraction; the approximate
// roots and reciprocals off by up to an ulp either way, as the hardware's may
// be), over boxes, triangles and hulls made to touch what decides them.
//
//   walk_bounds MODE COUNT SEED
//
// prints "cases N wrong W settled S": how many answers differ from the plain
// form, and how many the short cut settled by itself.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

static std::mt19937_64 rng;
static double uniform(double a, double b) { return a + (b - a) * ((double)(rng() >> 11) * 0x1p-53); }
static double spread(double a, double b) { return std::exp(uniform(std::log(a), std::log(b))); }
static uint32_t below(uint32_t n) { return (uint32_t)(rng() % n); }

static float off_by_an_ulp(float x) {
  const uint32_t k = below(3);
  return k == 0 ? x : std::nextafterf(x, k == 1 ? INFINITY : -INFINITY);
}
static float approximate_sqrt(float x) { return x == 0.0f ? 0.0f : off_by_an_ulp(std::sqrt(x)); }
static float approximate_rcp(float x) { return off_by_an_ulp(1.0f / x); }

#define __builtin_amdgcn_sqrtf approximate_sqrt
#define __builtin_amdgcn_rcpf approximate_rcp
#define __builtin_amdgcn_ballot_w64(p) ((unsigned long long)(p))
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, lane) (v)
#define __hip_atomic_fetch_add(p, v, order, scope) (*(p) += (v))
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __shfl_xor(v, off, width) (v)
#define atomicAdd(p, v) (*(p) += (v))
static struct {
  unsigned x;
} threadIdx;
static unsigned __float_as_uint(float f) {
  unsigned u;
  std::memcpy(&u, &f, 4);
  return u;
}
static float __uint_as_float(unsigned u) {
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
#include "cnq_walk.h"

using namespace cnq;

// ---- the plain forms (WGSL :234-255 and :519-574)
template <bool SKY>
static uint32_t plain_box(const Cone& c, f3 lo, f3 hi) {
  const uint32_t side = box_corners<SKY>(c, lo, hi);
  if (side == BOX_OUT) return BOX_OUT;
  return in_bound(c, (lo + hi) * 0.5f, 0.5f * len3(hi - lo)) ? side : BOX_OUT;
}

// A box's projected extent in bins.
static float plain_extent(const Cone& c, f3 lo, f3 hi) {
  const float g = (float)GRID;
  f2 a{3.4e38f, 3.4e38f}, b{-3.4e38f, -3.4e38f};
  for (uint32_t k = 0; k < 8; k++) {
    const f3 p = to_local(c, box_corner(lo, hi, k));
    const f2 q{(p.x / p.z - c.w0) / (c.w2 - c.w0) * g, (p.y / p.z - c.w1) / (c.w3 - c.w1) * g};
    a = f2{mn(a.x, q.x), mn(a.y, q.y)};
    b = f2{mx(b.x, q.x), mx(b.y, q.y)};
  }
  return mx(b.x - a.x, b.y - a.y);
}

// 0 culled, 1 a splat, 3 opened
template <bool SKY>
static uint32_t plain_node(const Cone& c, float prefilter, f3 lo, f3 hi) {
  const uint32_t side = plain_box<SKY>(c, lo, hi);
  if (side == BOX_OUT) return 0;
  return !(prefilter > 0.0f) || side != BOX_INSIDE || plain_extent(c, lo, hi) > prefilter ? 3 : 1;
}

// ---- inputs
struct Lanes {
  float cells[WALK_CELLS * 64], slots[POLY_SLOTS];
  Lane lane() { return Lane{cells, slots, POLY_STRIDE, ACC_CELLS, 0u}; }
};

static f3 any3(double s) { return f3{(float)uniform(-s, s), (float)uniform(-s, s), (float)uniform(-s, s)}; }
static f3 unit3() {
  for (;;) {
    const f3 v = any3(1.0);
    const float l = len3(v);
    if (l > 0.1f && l < 1.0f) return v / l;
  }
}

static LightCone light_cone(double shift) {
  for (;;) {
    LightRect r{};
    const f3 apex = any3(2.0) + f3{(float)shift, (float)-shift, 0.0f};
    const double far = spread(0.3, 300.0);
    const f3 at = apex + unit3() * (float)far;
    r.corner = {at.x, at.y, at.z, 0.0f};
    if (below(3) == 0) {
      r.corner.w = 2.0f;
      r.edge_u.x = (float)(far * spread(0.003, 0.9));
    } else {
      const f3 u = unit3() * (float)(far * spread(0.003, 3.0));
      const f3 v = norm3(cross3(u, unit3())) * (float)(far * spread(0.003, 3.0));
      r.edge_u = {u.x, u.y, u.z, 0.0f};
      r.edge_v = {v.x, v.y, v.z, 0.0f};
    }
    LightCone lc = light_cone_rect(apex, r, below(2) ? 2.0f : 8.0f);
    if (lc.ok) return lc;
  }
}

// The cone in the space of an object turned, scaled and moved at random.
static Cone in_object(const Cone& c) {
  const f3 a = unit3();
  const f3 b = norm3(cross3(a, unit3()));
  const f3 t = cross3(a, b);
  const float s = (float)spread(0.1, 10.0);
  const f3 o = c.apex + any3(30.0);
  const float xf[16] = {a.x, a.y, a.z, o.x, b.x, b.y, b.z, o.y, t.x, t.y, t.z, o.z, s, 1.0f / s, 0.0f, 0.0f};
  return cone_to_object(c, xf);
}

// A point on one of the planes that decide, or just anywhere in reach.
static f3 deciding_point(const Cone& c, double reach, bool sky) {
  const float z = (float)spread(reach * 1e-3, reach);
  float s = (float)uniform(-0.3, 1.3), t = (float)uniform(-0.3, 1.3);
  f3 p;
  switch (below(sky ? 8 : 7)) {
    case 0: s = 0.0f; break;
    case 1: s = 1.0f; break;
    case 2: t = 0.0f; break;
    case 3: t = 1.0f; break;
    case 4: {  // the far plane
      const f3 d = direction(c, s, t);
      const float k = (c.far_offset - dot3(c.far_normal, c.apex)) / dot3(c.far_normal, d);
      return c.apex + d * k;
    }
    case 5: return c.apex + c.right * (s * z) + c.up * (t * z) + c.forward * NEAR;
    case 7:  // the horizon
      p = any3(reach);
      return c.apex + (p - c.horizon * (dot3(p, c.horizon) / dot3(c.horizon, c.horizon)));
    default: break;
  }
  return c.apex + direction(c, s, t) * z;
}

static void any_box(const Cone& c, double reach, bool sky, f3& lo, f3& hi) {
  const f3 p = deciding_point(c, reach, sky);
  const double size = spread(reach * 1e-5, reach);
  const f3 e{(float)(below(8) ? uniform(0, size) : 0.0), (float)(below(8) ? uniform(0, size) : 0.0),
             (float)(below(8) ? uniform(0, size) : 0.0)};
  const uint32_t k = below(9);  // the point is a corner of the box, or lies inside it
  if (k == 8) {
    lo = p - e, hi = p + e;
    return;
  }
  lo = f3{(k & 1) ? p.x - e.x : p.x, (k & 2) ? p.y - e.y : p.y, (k & 4) ? p.z - e.z : p.z};
  hi = f3{(k & 1) ? p.x : p.x + e.x, (k & 2) ? p.y : p.y + e.y, (k & 4) ? p.z : p.z + e.z};
}

static void show(const char* what, uint32_t got, uint32_t want, const Cone& c, f3 lo, f3 hi) {
  std::printf("%s: %u, plain %u; apex %.9g %.9g %.9g horizon %.9g %.9g %.9g box %.9g %.9g %.9g .. %.9g %.9g %.9g\n", what,
              got, want, c.apex.x, c.apex.y, c.apex.z, c.horizon.x, c.horizon.y, c.horizon.z, lo.x, lo.y, lo.z, hi.x,
              hi.y, hi.z);
}

static uint64_t cases, wrong, settled;
static void note(const char* what, uint32_t got, uint32_t want, const Cone& c, f3 lo, f3 hi) {
  cases++;
  if (got == want) return;
  if (wrong++ < 3) show(what, got, want, c, lo, hi);
}

template <bool SKY>
static void check_box(const Cone& c, f3 lo, f3 hi) {
  static Lanes lanes;
  static float cov27[27];
  for (float& v : cov27) v = 1.0f;
  const ConeMargins cm = cone_margins(c);
  note("may_touch_box", may_touch_box<SKY>(c, cm, lo, hi), plain_box<SKY>(c, lo, hi) != BOX_OUT, c, lo, hi);
  BoxQuick b{};
  const uint32_t side = box_quick<SKY, true>(c, cm, lo, hi, b);
  if (side == BOX_OUT || (side != BOX_UNSURE && !b.bound_unsure)) settled++;
  // (a prefilter by the box's own extent too, a few ulps to either side)
  const float extent = plain_extent(c, lo, hi);
  const uint32_t k = below(8);
  const float prefilter = k == 0                            ? 0.0f
                          : k < 4                           ? (float)spread(0.05, 16.0)
                          : extent > 0.0f && extent < 1e30f ? extent * (1.0f + (float)uniform(-5e-7, 5e-7))
                                                            : 1.0f;
  Lane L = lanes.lane();
  // (with `hold` a splat is told and not drawn)
  const uint32_t test = node_cone_test<SKY>(c, cm, L, prefilter, lo, hi, cov27, true);
  note("node_cone_test", test == 0 || test == 3 ? test : 1, plain_node<SKY>(c, prefilter, lo, hi), c, lo, hi);
}

static void light_boxes(uint64_t n, bool objects) {
  for (uint64_t i = 0; i < n; i++) {
    const double shifts[4] = {0.0, 0.0, 1e3, 1e5};
    Cone c = light_cone(shifts[below(4)]).c;
    if (objects) c = in_object(c);
    const double reach = 1.5 * std::fabs(c.far_offset - dot3(c.far_normal, c.apex)) + 1e-3;
    for (int k = 0; k < 8; k++) {
      f3 lo, hi;
      any_box(c, reach, false, lo, hi);
      check_box<false>(c, lo, hi);
    }
  }
}

static void sky_boxes(uint64_t n) {
  for (uint64_t i = 0; i < n; i++) {
    const double shifts[3] = {0.0, 0.0, 1e3};
    const double shift = shifts[below(3)];
    const f3 normal = unit3() * (float)(below(2) ? 1.0 : spread(1e-3, 1e6));
    bool above;
    const Cone c = sky_face(below(6), any3(2.0) + f3{(float)shift, (float)-shift, 0.0f}, normal, below(8) != 0, above);
    const Cone o = below(4) == 0 ? in_object(c) : c;
    for (int k = 0; k < 8; k++) {
      f3 lo, hi;
      any_box(o, spread(0.1, 300.0), below(2) && o.horizon.x != 0.0f, lo, hi);
      check_box<true>(o, lo, hi);
    }
  }
}

// Boxes by an apex far from the origin, ulps to some hundreds of ulps wide.
static void apex_boxes(uint64_t n) {
  for (uint64_t i = 0; i < n; i++) {
    const double at = spread(1.0, 1e6);
    const Cone c = light_cone(at).c;
    const double ulp = at * 0x1p-23, size = below(2) ? 4.0 : 100.0;
    for (int k = 0; k < 8; k++) {
      f3 lo, hi;
      auto axis = [&](float x, float& a, float& b) {
        const double step = std::fabs(x) < 4.0 && below(2) ? spread(1e-4, 1.0) / size : ulp;
        a = (float)(x + uniform(-size, size) * step);
        b = (float)(a + (below(4) ? uniform(0, size) * step : 0.0));
      };
      axis(c.apex.x, lo.x, hi.x), axis(c.apex.y, lo.y, hi.y), axis(c.apex.z, lo.z, hi.z);
      check_box<false>(c, lo, hi);
    }
  }
}

// Cones of any window and far plane (a lattice cone's is its light's, not its
// forward axis), at any scale, and boxes that are points, empty, unbounded or
// not a number.
static void any_boxes(uint64_t n) {
  for (uint64_t i = 0; i < n; i++) {
    Cone c{};
    c.apex = any3(spread(1e-6, 1e8));
    c.forward = unit3();
    c.right = norm3(cross3(c.forward, unit3()));
    c.up = cross3(c.forward, c.right);
    const float u = (float)(uniform(-1, 1) * spread(1e-3, 1e4)), v = (float)(uniform(-1, 1) * spread(1e-3, 1e4));
    const float eu = (float)spread(1e-6, 1e2), ev = (float)spread(1e-6, 1e2);
    c.w0 = u - eu, c.w2 = u + eu, c.w1 = v - ev, c.w3 = v + ev;
    c.far_normal = below(2) ? c.forward : unit3();
    const double far = spread(1e-6, 1e8);
    c.far_offset = dot3(c.far_normal, c.apex) + (float)far;
    bound_cone(c, norm3(direction(c, 0.5f, 0.5f)));
    for (int k = 0; k < 8; k++) {
      f3 lo, hi;
      any_box(c, below(2) ? far : spread(1e-8, 1e12), false, lo, hi);
      switch (below(40)) {
        case 0: hi.x = INFINITY; break;
        case 1: lo.y = -INFINITY, hi.y = INFINITY; break;
        case 2: hi = lo; break;
        case 3: lo = f3{3.4e38f, 3.4e38f, 3.4e38f}, hi = -lo; break;
        case 4: hi.z = NAN; break;
        case 5: lo.x = -1e38f, hi.x = 1e38f; break;
        case 6: lo = hi = c.apex; break;
        default: break;
      }
      check_box<false>(c, lo, hi);
    }
  }
}

// ---- draws: the accumulator after a draw in LDS and after the general clips
static void note_draw(bool a, bool b, Lanes& x, Lanes& y) {
  cases++;
  bool same = a == b;
  for (uint32_t k = 0; k < ACC_CELLS; k++) same = same && std::memcmp(&x.cells[64 * k], &y.cells[64 * k], 4) == 0;
  if (!same && wrong++ < 3) std::printf("a draw differs from the general clips\n");
}

static void triangles(uint64_t n) {
  static Lanes x, y;
  for (uint64_t i = 0; i < n; i++) {
    const double shifts[3] = {0.0, 0.0, 1e3};
    Cone c = light_cone(shifts[below(3)]).c;
    if (below(2)) c = in_object(c);
    const double reach = std::fabs(c.far_offset - dot3(c.far_normal, c.apex));
    for (int k = 0; k < 4; k++) {
      const f3 at = deciding_point(c, reach, false);
      const double size = spread(reach * 1e-4, reach * 4);
      f3 v[3];
      for (f3& p : v) p = below(4) ? at + any3(size) : deciding_point(c, reach, false);
      if (below(16) == 0) v[2] = v[1];
      const float weight = below(2) ? 1.0f : 0.37f;
      Lane L = x.lane();
      clear_acc(L);
      const bool drawn = rasterize(c, L, v[0], v[1], v[2], weight);
      Lane G = y.lane();
      clear_acc(G);
      const float su = (float)GRID / (c.w2 - c.w0), sv = (float)GRID / (c.w3 - c.w1);
      auto past = [&](f3 p) { return c.far_offset - dot3(c.far_normal, p) < 0.0f; };
      const f3 l0 = to_local(c, v[0]), l1 = to_local(c, v[1]), l2 = to_local(c, v[2]);
      uint32_t slot = Q2A;
      bool grid_clip = false, plain = false;
      uint32_t m = general_polygon(c, G, v[0], v[1], v[2], past(v[0]) || past(v[1]) || past(v[2]), l0, l1, l2, su, sv,
                                   slot, grid_clip);
      if (grid_clip) m = clip_to_grid(G, slot, m);
      if (m >= 3) {
        plain = true;
        for (uint32_t e = 0; e < m; e++)
          draw_edge(G, clamp_grid(G.p2(slot, e)), clamp_grid(G.p2(slot, e + 1 < m ? e + 1 : 0)), weight);
      }
      settled += l0.z >= NEAR && l1.z >= NEAR && l2.z >= NEAR && !(past(v[0]) || past(v[1]) || past(v[2]));
      note_draw(drawn, plain, x, y);
    }
  }
}

static void hulls(uint64_t n) {
  static Lanes x, y;
  for (uint64_t i = 0; i < n; i++) {
    f2 p[8];
    const double size = spread(0.01, 12.0);
    const f2 at{(float)uniform(-2, 10), (float)uniform(-2, 10)};
    const bool grid = below(4) == 0;  // corners on the grid's own lines
    for (f2& q : p) {
      q = f2{at.x + (float)uniform(-size, size), at.y + (float)uniform(-size, size)};
      if (grid) q = f2{std::round(q.x), std::round(q.y)};
    }
    Lane L = x.lane();
    clear_acc(L);
    const bool drawn = draw_hull(L, p, 0.7f);
    Lane G = y.lane();
    clear_acc(G);
    f2 last{0.0f, 0.0f};
    uint32_t m = hull8(G, p, last);
    for (uint32_t e = 0; e < m; e++) G.put2(Q2A, e, e < GRID_VERTS ? G.vert(e) : last);
    uint32_t slot = Q2A;
    m = clip_to_grid(G, slot, m);
    const bool plain = m >= 3;
    for (uint32_t e = 0; plain && e < m; e++)
      draw_edge(G, clamp_grid(G.p2(slot, e)), clamp_grid(G.p2(slot, e + 1 < m ? e + 1 : 0)), 0.7f);
    settled += m <= GRID_VERTS;
    note_draw(drawn, plain, x, y);
  }
}

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const char* mode = argv[1];
  const uint64_t n = std::strtoull(argv[2], nullptr, 10);
  rng.seed(std::strtoull(argv[3], nullptr, 10));
  if (!std::strcmp(mode, "light"))
    light_boxes(n, false);
  else if (!std::strcmp(mode, "object"))
    light_boxes(n, true);
  else if (!std::strcmp(mode, "sky"))
    sky_boxes(n);
  else if (!std::strcmp(mode, "apex"))
    apex_boxes(n);
  else if (!std::strcmp(mode, "any"))
    any_boxes(n);
  else if (!std::strcmp(mode, "triangle"))
    triangles(n);
  else if (!std::strcmp(mode, "hull"))
    hulls(n);
  else
    return 2;
  std::printf("cases %llu wrong %llu settled %llu\n", (unsigned long long)cases, (unsigned long long)wrong,
              (unsigned long long)settled);
  return 0;
}
