// Device geometry of the bake: the visibility predicate and the
// point-to-patch solid angle, in float64.
//
// The predicate reproduces geometry._basic_visibility /
// _point_in_polygon / _project_to_plane / _rotation_matrix
// (sparrowpy/geometry.py:498-686, 841-909) operation for operation, so the
// boolean results are the reference's bits.  Three things differ in
// organisation only, never in result:
//  * Everything that depends on the blocking polygon alone (rotation rows,
//    rotated corners, edge normals and lengths, the rotated bounding box)
//    is computed once per polygon into a BlockerRec instead of once per
//    query.
//  * Work whose outcome is already decided is skipped: the winding test is
//    not run for a point more than 1e-3 outside the polygon's bounding box
//    in the rotated frame (the reference's edge test only accepts crossing
//    points within ~1e-6 of an edge, so its count is 0 there), and the
//    "segment crosses the polygon" test evaluates the cheap
//    (pt - a).(pt - b) < 0 condition before the winding test (both are pure
//    and are combined with AND).
//  * Blockers that cannot block a segment are not evaluated for it: groups
//    of coplanar blockers are dropped for a tile of segments
//    (may_block_tile) and for one segment (sight, may_block), and so are
//    the members of a group.
#pragma once

#include "spr_common.hpp"

namespace spr {

constexpr double kEta = 1e-6;        // geometry.py:616, 845
constexpr double kBoxMargin = 1e-3;  // >> kEta, see header comment

struct BlockerRec {
  double n[3];      // plane normal
  double p0[3];     // first corner
  double m0[3];     // rotation matrix row 0 (normal -> +z)
  double m1[3];     // rotation matrix row 1
  double px[4];     // rotated corners, x
  double py[4];     // rotated corners, y
  double nlx[4];    // edge normals (-side.y, side.x) / |side|
  double nly[4];
  double elen[4];   // |a1 - a0|
  double box[4];    // xmin, xmax, ymin, ymax of the rotated corners
};
static_assert(sizeof(BlockerRec) == 36 * sizeof(double), "BlockerRec size");

// geometry.py:498-559 _rotation_matrix(n_in) with n_out = (0, 0, 1);
// only rows 0 and 1 are used (projection to the plane's 2-D frame).
__host__ __device__ inline void rotation_rows(const double *n_in,
                                              double *m0, double *m1) {
  const double n_out[3] = {0.0, 0.0, 1.0};
  int counter = 0;
  for (int i = 0; i < 3; ++i)
    if (n_in[i] == n_out[i]) counter += 1;
  double m[3][3];
  if (counter == 3) {
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) m[i][j] = (i == j) ? 1.0 : 0.0;
  } else {
    d3 nv{n_in[0], n_in[1], n_in[2]};
    double na = norm(nv);
    d3 a{n_in[0] / na, n_in[1] / na, n_in[2] / na};
    d3 ov{n_out[0], n_out[1], n_out[2]};
    double nb = norm(ov);
    d3 b{n_out[0] / nb, n_out[1] / nb, n_out[2] / nb};
    double c = dot(a, b);
    if (c != -1.0) {
      d3 v = cross(a, b);
      double s = norm(v);
      double k[3][3] = {{0.0, -v.z, v.y}, {v.z, 0.0, -v.x}, {-v.y, v.x, 0.0}};
      double f = (1.0 - c) / (s * s);
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
          double kk =
              (k[i][0] * k[0][j] + k[i][1] * k[1][j]) + k[i][2] * k[2][j];
          double e = (i == j) ? 1.0 : 0.0;
          m[i][j] = (e + k[i][j]) + kk * f;
        }
    } else {
      const double r[3][3] = {{-1., 0., 0.}, {0., 1., 0.}, {0., 0., -1.}};
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) m[i][j] = r[i][j];
    }
  }
  for (int j = 0; j < 3; ++j) {
    m0[j] = m[0][j];
    m1[j] = m[1][j];
  }
}

// Up to kGroup consecutive blockers in one plane: their normals, and with
// them the rotation rows, are the same bits, and their planes' offsets
// follow one another within kPlaneStep (1 + |c|).
constexpr int kGroup = 32;
constexpr double kPlaneStep = 1e-12;
constexpr double kLongEdge = 1e3;  // see may_block
constexpr int kLines = 36;         // 33 rows of corners, with some to spare
constexpr double kLineStep = 1e-6;
// Corners left out of a group's lines follow from one to the next within
// kLineStep, so one of the lines is within this of each.
constexpr double kLineSlack = 4 * kGroup * kLineStep;
constexpr double kFarStep = 1e30;
struct BlockerGroup {
  double n[3], m0[3], m1[3];
  double c;         // n . p0 of the first member
  double dc;        // no member's offset is further from c
  double box[4];    // union of the members' boxes
  int32_t count;
  int32_t left;     // 1: no edge longer than kLongEdge (see may_block)
  int32_t n_lines;  // 0: more than kLines
  // The lines as y0 + k step (k whole), each within kLineSlack: most walls'
  // patches.  step 0: they are not; a single line has a step out of reach.
  double y0, step, inv_step;
  // rotated y of the members' corners, those within kLineStep once
  double lines[kLines];
};

// geometry.py:614-686 _point_in_polygon for a 4-corner blocker.
__host__ __device__ inline bool point_in_blocker(d3 p, const BlockerRec &r) {
  if (fabs(dot(p - load3(r.p0), load3(r.n))) > kEta) return false;
  d2 pt{dot(load3(r.m0), p), dot(load3(r.m1), p)};
  // Bounding-box early out (see header comment): count stays 0.
  if (pt.x > r.box[1] + kBoxMargin || pt.y < r.box[2] - kBoxMargin ||
      pt.y > r.box[3] + kBoxMargin)
    return false;
  int count = 0;
  const d2 ptp{pt.x + 1.0, pt.y + 0.0};
  const d2 v = ptp - pt;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const d2 a1{r.px[(i + 1) & 3], r.py[(i + 1) & 3]};
    const d2 a0{r.px[i], r.py[i]};
    const d2 nl{r.nlx[i], r.nly[i]};
    double dotprod = dot(v, nl);
    if (!(fabs(dotprod) > 1e-6)) continue;
    d2 w = ptp - a1;
    double fac = -(dot(nl, w) / dotprod);
    d2 b{(w.x + a1.x) + fac * v.x, (w.y + a1.y) + fac * v.y};
    if (b.x > pt.x) {
      if (fabs((norm(b - a0) + norm(b - a1)) - r.elen[i]) <= kEta) {
        double dd = dot(b - pt, nl);
        if (dd > 0)
          count += 1;
        else if (dd < 0)
          count -= 1;
      }
    }
  }
  return count != 0;
}

// Culling that keeps basic_visibility's result.  The predicate can only
// return "blocked" for a segment a-b if a point of it (an endpoint, or the
// crossing point, which lies on the segment up to rounding) passes
// point_in_blocker: within kEta of the plane, at rotated x <= box[1] +
// kBoxMargin and rotated y within box[2..3] +- kBoxMargin.  Such points lie
// on the part of the segment within kCullPlane of the plane, and the
// rotated x and y are linear along it, so a blocker whose accepted x / y
// range that part misses by more than kCullBox leaves the pair visible --
// as does a blocker whose plane the segment never comes within kCullPlane
// of.  The margins exceed the thresholds by far more than any rounding of
// points on the segment.
constexpr double kCullPlane = 1e-3;  // >> kEta
constexpr double kCullBox = 2e-3;    // > kBoxMargin

// Interval bounds of the linear form c.p over the axis-aligned box [lo, hi].
__device__ inline double form_min(d3 c, d3 lo, d3 hi) {
  return (fmin(c.x * lo.x, c.x * hi.x) + fmin(c.y * lo.y, c.y * hi.y)) +
         fmin(c.z * lo.z, c.z * hi.z);
}
__device__ inline double form_max(d3 c, d3 lo, d3 hi) {
  return (fmax(c.x * lo.x, c.x * hi.x) + fmax(c.y * lo.y, c.y * hi.y)) +
         fmax(c.z * lo.z, c.z * hi.z);
}

// For every segment from a point of box I to a point of box J.  If one box
// lies within kCullPlane of the plane and the other beyond it (a patch's
// own wall seen from off the wall), the part of each segment within
// kCullPlane of the plane stays within tau * L of the first box, with
// tau = 2 kCullPlane / (gap - kCullPlane) and L the longest segment, so
// only that neighbourhood of the box is tested; otherwise the whole union
// box is.
__device__ inline bool may_block_tile(d3 ilo, d3 ihi, d3 jlo, d3 jhi,
                                      const BlockerGroup &r) {
  const d3 n = load3(r.n), m0 = load3(r.m0), m1 = load3(r.m1);
  const double np0 = r.c;
  const double di0 = form_min(n, ilo, ihi) - np0;
  const double di1 = form_max(n, ilo, ihi) - np0;
  const double dj0 = form_min(n, jlo, jhi) - np0;
  const double dj1 = form_max(n, jlo, jhi) - np0;
  if ((di0 > kCullPlane && dj0 > kCullPlane) ||
      (di1 < -kCullPlane && dj1 < -kCullPlane))
    return false;
  const d3 ulo{fmin(ilo.x, jlo.x), fmin(ilo.y, jlo.y), fmin(ilo.z, jlo.z)};
  const d3 uhi{fmax(ihi.x, jhi.x), fmax(ihi.y, jhi.y), fmax(ihi.z, jhi.z)};
  d3 lo = ulo, hi = uhi;
  double grow = 0.0;
  const bool i_on = di0 >= -kCullPlane && di1 <= kCullPlane;
  const bool j_on = dj0 >= -kCullPlane && dj1 <= kCullPlane;
  const double gap_j = fmax(dj0, -dj1), gap_i = fmax(di0, -di1);
  if (i_on && !j_on && gap_j > 2 * kCullPlane) {
    lo = ilo, hi = ihi;
    grow = 2 * kCullPlane / (gap_j - kCullPlane) * norm(uhi - ulo);
  } else if (j_on && !i_on && gap_i > 2 * kCullPlane) {
    lo = jlo, hi = jhi;
    grow = 2 * kCullPlane / (gap_i - kCullPlane) * norm(uhi - ulo);
  }
  if (form_min(m0, lo, hi) - grow > r.box[1] + kCullBox) return false;
  return !(form_max(m1, lo, hi) + grow < r.box[2] - kCullBox ||
           form_min(m1, lo, hi) - grow > r.box[3] + kCullBox);
}

// Where one segment can meet the plane of a group: every point of it that
// the predicate could find in a member lies within g of (x, y) in the
// rotated frame, or of (x2, y2) if two is set.
struct Sight {
  double x, y, g, x2, y2;
  bool two;
};

// a . b as the culls form it, two fused steps (their margins cover rounding;
// the predicate's dot() is the reference's).
__host__ __device__ inline double cull_dot(d3 a, d3 b) {
  return fma(a.z, b.z, fma(a.y, b.y, a.x * b.x));
}

// 1 / x to about 1e-15 of it (hardware reciprocal and a Newton step); what
// overflows or is 0 gives an infinity or NaN, which no cull drops.
__host__ __device__ inline double cull_inverse(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(x);
  return fma(fma(-x, r, 1.0), r, r);
#else
  return 1.0 / x;
#endif
}

// False if the segment a-b cannot be blocked by any member: both ends lie
// beyond kCullPlane on one side, so that neither is in the plane and the
// crossing point lies outside the segment.  With the ends beyond kCullPlane
// on either side only the crossing point counts (a member's plane, up to dc off
// this one, moves it by g); with one end near the plane
// only that end's neighbourhood (as in may_block_tile); with both ends near
// the plane and the segment as good as parallel to it (the reference takes no
// crossing point below 1e-6) only the two ends; otherwise the whole segment.
// A NaN anywhere makes the later comparisons false, and members are kept.
__host__ __device__ inline bool sight(d3 a, d3 b, const BlockerGroup &r,
                                      Sight &s) {
  const d3 n = load3(r.n), m0 = load3(r.m0), m1 = load3(r.m1);
  const double da = cull_dot(n, a) - r.c, db = cull_dot(n, b) - r.c;
  if ((da > kCullPlane && db > kCullPlane) ||
      (da < -kCullPlane && db < -kCullPlane))
    return false;
  const double xa = cull_dot(m0, a), ya = cull_dot(m1, a);
  const double xb = cull_dot(m0, b), yb = cull_dot(m1, b);
  const bool na = fabs(da) <= kCullPlane, nb = fabs(db) <= kCullPlane;
  s.two = false;
  s.g = 0.0;
  if (!na && !nb) {
    const double inv = cull_inverse(da - db), t = da * inv;
    s.x = fma(t, xb - xa, xa);
    s.y = fma(t, yb - ya, ya);
    s.g = r.dc * (fabs(xb - xa) + fabs(yb - ya)) * fabs(inv);
    return true;
  }
  if (na && fabs(db) > 2 * kCullPlane) {
    s.x = xa, s.y = ya;
    s.g = 2 * kCullPlane / (fabs(db) - kCullPlane) * norm(b - a);
  } else if (nb && fabs(da) > 2 * kCullPlane) {
    s.x = xb, s.y = yb;
    s.g = 2 * kCullPlane / (fabs(da) - kCullPlane) * norm(b - a);
  } else if (fabs(da - db) < 5e-7) {
    s.x = xa, s.y = ya, s.x2 = xb, s.y2 = yb;
    s.two = true;
  } else {
    s.x = xa, s.y = ya;
    s.g = norm(b - a);
  }
  return true;
}

// Whether a point within g of (x, y) may pass point_in_blocker with this box:
// it needs x <= box[1] and y in box[2..3], up to the margin.
__host__ __device__ inline bool in_reach(double x, double y, double g,
                                         const double *box) {
  return ((int)(x - g > box[1] + kCullBox) | (int)(y + g < box[2] - kCullBox) |
          (int)(y - g > box[3] + kCullBox)) == 0;
}

// The same for one member, which also drops points left of its box: their
// ray (to +x) crosses as many edges upwards as downwards, so the count is 0,
// unless it passes a corner so closely that the edge test's tolerance
// decides.  More than kCullBox in y from every corner, a crossed edge spans
// at least twice that in y, so with edges up to kLongEdge its normal's x is
// above the 1e-6 at which the reference skips an edge, and both the edge
// test and the sign of each crossing are decided far above rounding.
__host__ __device__ inline bool left_of(double x, double g, double x_min) {
  return x + (kCullBox + g) < x_min;
}
// Whether y is that close to one of the group's lines of corners.
__host__ __device__ inline bool near_line(double y, double g,
                                          const BlockerGroup &r) {
  const double m = kCullBox + 2 * kLineSlack + g;
  if (r.step > 0) {  // uniform
    const double u = (y - r.y0) * r.inv_step;
    return !(fabs(u - rint(u)) * r.step > m);
  }
  bool near = false;
  for (int l = 0; l < r.n_lines; ++l) near |= !(fabs(y - r.lines[l]) > m);
  return near;
}
__host__ __device__ inline bool may_block(double x, double y, double g,
                                          int left, const BlockerRec &r) {
  const double m = kCullBox + g;
  int near = left == 0 || !left_of(x, g, r.box[0]);
  for (int q = 0; q < 4; ++q) near |= !(fabs(y - r.py[q]) > m);
  return (in_reach(x, y, g, r.box) & near) != 0;
}

// geometry.py:841-909 _basic_visibility(vis_point=a, eval_point=b).
__host__ __device__ inline bool basic_visibility(d3 a, d3 b,
                                                 const BlockerRec &r) {
  const bool vin = point_in_blocker(a, r);
  const bool ein = point_in_blocker(b, r);
  const d3 n = load3(r.n);
  if (!vin && !ein) {
    // _project_to_plane(origin=a, point=b, plane_pt=p0, normal=n,
    //                   check_normal=False)
    d3 v = b - a;
    double dotprod = dot(v, n);
    if (fabs(dotprod) > 1e-6) {
      const d3 p0 = load3(r.p0);
      d3 w = b - p0;
      double fac = -(dot(n, w) / dotprod);
      d3 pt{(w.x + p0.x) + fac * v.x, (w.y + p0.y) + fac * v.y,
            (w.z + p0.z) + fac * v.z};
      if (dot(pt - a, pt - b) < 0 && point_in_blocker(pt, r)) return false;
    }
    return true;
  }
  if (vin && !ein && dot(n, b - a) < 0) return false;
  if (!vin && ein && dot(n, a - b) < 0) return false;
  const d3 p0 = load3(r.p0);
  if (fabs(dot(a - p0, n)) < kEta && fabs(dot(b - p0, n)) < kEta &&
      (vin || ein))
    return false;
  return true;
}

// geometry.py:688-715 _sphere_tangent_vector
__device__ inline d3 sphere_tangent(d3 v0, d3 v1) {
  if (fabs(dot(v0, v1)) > 1e-10) {
    d3 d = v1 - v0;
    double s = dot(d, v0) / dot(v0, v0);
    d3 o{d.x - s * v0.x, d.y - s * v0.y, d.z - s * v0.z};
    return div(o, norm(o));
  }
  return div(v1, norm(v1));
}

// geometry.py:420-440 _polygon_area (4 corners)
__device__ inline double quad_area(const double *pts) {
  double area = 0.0;
  d3 p0 = load3(pts);
  for (int t = 0; t < 2; ++t) {
    d3 c = cross(load3(pts + 3 * (t + 1)) - p0, load3(pts + 3 * (t + 2)) - p0);
    area += 0.5 * norm(c);
  }
  return area;
}

// integration.py:295-344 pt_solution for a 4-corner patch;
// receiver: divide by pi*area, source: by pi*4.
__device__ inline double pt_solution(d3 point, const double *pts,
                                     bool receiver) {
  double area = receiver ? quad_area(pts) : 4.0;
  d3 on[4];
  for (int i = 0; i < 4; ++i) {
    d3 d = load3(pts + 3 * i) - point;
    on[i] = div(d, norm(d));
  }
  double sum = 0.0;
  for (int i = 0; i < 4; ++i) {
    d3 t0 = sphere_tangent(on[i], on[(i + 3) & 3]);
    d3 t1 = sphere_tangent(on[i], on[(i + 1) & 3]);
    sum += acos(dot(t0, t1));
  }
  double factor = sum - 2.0 * M_PI;
  return factor / (M_PI * area);
}

}  // namespace spr
