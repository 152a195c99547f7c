// Bake kernels: visibility, visible-pair list, universal form factors,
// outgoing-direction maps, the dense directional form factor and source
// injection.  All geometry is float64 (see spr_common.hpp on rounding).
//
// Reference: sparrowpy/geometry.py (visibility), sparrowpy/form_factor/
// universal.py and integration.py (form factors, point-patch factors),
// sparrowpy/classes/RadiosityFast.py (bake_geometry, init_source_energy).
#include "spr_common.hpp"
#include "spr_fft.hpp"
#include "spr_geom.hpp"
#include "spr_util.hpp"

namespace spr {
namespace {

// ---------------------------------------------------------------------
// visibility
// ---------------------------------------------------------------------
// Members of the group that starts at bit m, of n_here blockers in its run.
__device__ inline int count_of_group(uint32_t head, int m, int n_here) {
  const uint32_t later = m + 1 < kGroup ? head >> (m + 1) : 0u;
  return later ? __ffs((int)later) : n_here - m;
}

// Component q of the box (xmin, xmax, ymin, ymax) of corners from..to-1.
__device__ inline double extent(const double *sx, const double *sy, int from,
                                int to, int q) {
  const double *v = q < 2 ? sx : sy;
  double e = v[from];
#pragma unroll 8
  for (int t = from + 1; t < to; ++t)
    e = (q & 1) ? fmax(e, v[t]) : fmin(e, v[t]);
  return e;
}

// Blocker records, and the groups of coplanar blockers among each kGroup
// consecutive ones: bit m of heads[k / kGroup] is set where blocker k's run
// of kGroup starts a group, and groups[] holds the group at the index of its
// first member.  A workgroup per run, a lane per corner: most calls have a
// handful of blockers and wait for the kernel's own code to come in from
// memory, so every step is written once and not unrolled over corners (6
// walls 5 us, 208 patches 11 us; a lane per blocker 19 us for either).
__global__ __launch_bounds__(4 * kGroup) void blocker_kernel(
    int64_t NS, const double *__restrict__ normals,
    const double *__restrict__ pts, BlockerRec *__restrict__ recs,
    BlockerGroup *__restrict__ groups, uint32_t *__restrict__ heads) {
  __shared__ double sx[4 * kGroup], sy[4 * kGroup];
  __shared__ uint32_t s_head, s_long, s_lines[kGroup];
  const int t = (int)threadIdx.x, m = t >> 2, q = t & 3;
  const int64_t k0 = (int64_t)blockIdx.x * kGroup, k = k0 + m;
  const int n_here = (int)(NS - k0 < kGroup ? NS - k0 : kGroup);
  const bool valid = m < n_here;
  if (t < kGroup) s_lines[t] = 0;
  if (t == 0) s_head = s_long = 0;
  double m0[3], m1[3];
  d3 n{0.0, 0.0, 0.0}, p0{0.0, 0.0, 0.0};
  double c = 0.0;
  bool same = false;  // in the plane of the blocker before
  if (valid) {
    n = load3(normals + 3 * k);
    p0 = load3(pts + 12 * k);
    c = dot(n, p0);
    if (m > 0) {
      const d3 o = load3(normals + 3 * (k - 1));
      const double co = dot(n, load3(pts + 12 * (k - 1)));
      same = __double_as_longlong(o.x) == __double_as_longlong(n.x) &&
             __double_as_longlong(o.y) == __double_as_longlong(n.y) &&
             __double_as_longlong(o.z) == __double_as_longlong(n.z) &&
             fabs(c - co) <= kPlaneStep * (1.0 + fabs(c));
    }
    rotation_rows(normals + 3 * k, m0, m1);
    const d3 p = load3(pts + 12 * k + 3 * q);
    sx[t] = dot(load3(m0), p);
    sy[t] = dot(load3(m1), p);
  }
  __syncthreads();
  if (valid) {
    BlockerRec &r = recs[k];
    const int t1 = (t & ~3) | ((q + 1) & 3);
    const d2 side = d2{sx[t1], sy[t1]} - d2{sx[t], sy[t]};
    const double ns = norm(side);
    r.px[q] = sx[t], r.py[q] = sy[t];
    r.nlx[q] = -side.y / ns;
    r.nly[q] = side.x / ns;
    r.elen[q] = ns;
    // n, p0, m0, m1: three components each, a row to a lane
    double *row = q == 0 ? r.n : q == 1 ? r.p0 : q == 2 ? r.m0 : r.m1;
    row[0] = q == 0 ? n.x : q == 1 ? p0.x : q == 2 ? m0[0] : m1[0];
    row[1] = q == 0 ? n.y : q == 1 ? p0.y : q == 2 ? m0[1] : m1[1];
    row[2] = q == 0 ? n.z : q == 1 ? p0.z : q == 2 ? m0[2] : m1[2];
    r.box[q] = extent(sx, sy, t & ~3, (t & ~3) + 4, q);
    if (!(ns <= kLongEdge)) atomicOr(&s_long, 1u << m);
    if (q == 0 && !same) atomicOr(&s_head, 1u << m);
  }
  __syncthreads();
  const uint32_t head = s_head;
  if (t == 0) heads[blockIdx.x] = head;
  const int start =
      31 - __clz((int)(head & (uint32_t)((2ull << m) - 1ull)));
  const int count = count_of_group(head, start, n_here);
  if (valid) {
    // a line for a corner whose y no earlier corner of the group has
    bool first = true;
#pragma unroll 4
    for (int e = 4 * start; e < t; ++e)
      first &= !(fabs(sy[t] - sy[e]) <= kLineStep);
    if (first) {
      const uint32_t l = atomicAdd(&s_lines[start], 1u);
      if (l < kLines) groups[k0 + start].lines[l] = sy[t];
    }
  }
  __syncthreads();
  const int n_lines = (int)s_lines[m] <= kLines ? (int)s_lines[m] : 0;
  if (!valid || same) return;
  BlockerGroup &g = groups[k];
  const double u = extent(sx, sy, 4 * m, 4 * (m + count), q);
  g.box[q] = u;
  // evenly spaced lines?  (the member's four lanes look at a corner each)
  const double y0 = __shfl(u, (t & 60) | 2), y1 = __shfl(u, (t & 60) | 3);
  const double step = n_lines > 1 ? (y1 - y0) / (n_lines - 1) : kFarStep;
  const double inv = 1.0 / step;
  bool even = n_lines > 0;
#pragma unroll 4
  for (int e = m; e < m + count; ++e) {
    const double l = (sy[4 * e + q] - y0) * inv;
    even &= fabs(l - rint(l)) * step <= kLineSlack;
  }
  even = (__ballot(even) >> (t & 60) & 15u) == 15u;
  if (q != 0) return;
  g.n[0] = n.x, g.n[1] = n.y, g.n[2] = n.z;
  for (int e = 0; e < 3; ++e) g.m0[e] = m0[e], g.m1[e] = m1[e];
  g.c = c;
  g.dc = kGroup * kPlaneStep * (2.0 + fabs(c));
  g.count = count;
  g.left = (s_long >> m & ((2u << (count - 1)) - 1u)) == 0;
  g.n_lines = n_lines;
  g.y0 = y0;
  g.inv_step = inv;
  g.step = even ? step : 0.0;
}

// Whether any member of the group that starts at blocker k0 blocks this
// lane's segment a-b.  Every lane marks the members that its segment can meet
// (records through scalar loads), then evaluates the predicate for its own
// marks: nearly always one or two, so a wave takes a few turns instead of one
// for each member that any of its lanes meets.
__device__ inline bool group_blocks(d3 a, d3 b, bool alive, int64_t k0,
                                    const BlockerGroup &grp,
                                    const BlockerRec *__restrict__ recs) {
  Sight s;
  bool meets = alive && sight(a, b, grp, s);
  if (!__any(meets)) return false;
  if (!meets) s = Sight{0.0, 0.0, 0.0, 0.0, 0.0, false};
  if (!s.two) s.x2 = s.x, s.y2 = s.y;
  const bool any_two = __any(s.two);
  meets = meets && (in_reach(s.x, s.y, s.g, grp.box) ||
                    in_reach(s.x2, s.y2, s.g, grp.box));
  const bool left = meets && left_of(s.x, s.g, grp.box[0]) &&
                    left_of(s.x2, s.g, grp.box[0]);
  if (grp.left != 0 && grp.n_lines > 0 && __any(left)) {
    bool near = near_line(s.y, s.g, grp);
    if (any_two) near |= near_line(s.y2, s.g, grp);
    meets = meets && (near || !left);
  }
  if (!__any(meets)) return false;
  uint32_t mine = 0;
#pragma unroll 4
  for (int m = 0; m < grp.count; ++m) {
    const BlockerRec &r = recs[k0 + m];
    mine |= (uint32_t)may_block(s.x, s.y, s.g, grp.left, r) << m;
  }
  if (any_two)
    for (int m = 0; m < grp.count; ++m)
      mine |= (uint32_t)may_block(s.x2, s.y2, s.g, grp.left, recs[k0 + m])
              << m;
  if (!meets) mine = 0;
  bool blocked = false;
  while (mine != 0 && !blocked) {
    blocked = !basic_visibility(a, b, recs[k0 + __ffs((int)mine) - 1]);
    mine &= mine - 1;
  }
  return blocked;
}

// Thread per pair (i, j) of a 16x16 tile.  The workgroup first culls the
// groups of blockers for the whole tile (may_block_tile over the boxes of its
// 16 row and 16 column patch centres) into a candidate list in LDS; every
// lane then walks the candidates (a uniform loop) until its pair is blocked.
// Culls and marks only drop blockers that cannot block the pair, so the flags
// are those of the full scan.
// Bound by sight()'s float64 arithmetic and by the wait for each group's
// record: in a canyon of 5,122 patches, all of them blockers, a wave looks at
// 86 groups, meets the box of 2.6 and takes 1.7 turns of the predicate, in
// 5.6 ms for 13.1 M pairs (8.0 with unfused products, a division per group
// and each line of corners compared); testing the predicate for every blocker that the
// tile's cull leaves (about 1,500) took 105 ms.
__global__ __launch_bounds__(256, 4) void p2p_visibility_kernel(
    int64_t P, const double *__restrict__ centers, int64_t NS,
    const BlockerRec *__restrict__ recs,
    const BlockerGroup *__restrict__ groups,
    const uint32_t *__restrict__ heads, uint8_t *__restrict__ vis) {
  __shared__ int32_t cand[256];
  __shared__ int32_t wave_count[4];
  __shared__ double box[12];
  const int64_t ti = blockIdx.y, tj = blockIdx.x;
  const int64_t i = ti * 16 + (threadIdx.x >> 4);
  const int64_t j = tj * 16 + (threadIdx.x & 15);
  if (ti > tj) {  // tile entirely below the diagonal
    if (i < P && j < P) vis[i * P + j] = 0;
    return;
  }
  const bool valid = i < P && j < P;
  bool alive = valid && i < j;
  d3 a{0, 0, 0}, b{0, 0, 0};
  if (alive) {
    a = load3(centers + 3 * i);
    b = load3(centers + 3 * j);
  }
  if (threadIdx.x < 2) {
    // bounding box of the tile's row (i) or column (j) patch centres
    const int64_t t = threadIdx.x == 0 ? ti : tj;
    d3 lo{INFINITY, INFINITY, INFINITY}, hi{-INFINITY, -INFINITY, -INFINITY};
    for (int q = 0; q < 16; ++q) {
      const int64_t k = t * 16 + q;
      if (k >= P) break;
      const d3 c = load3(centers + 3 * k);
      lo = d3{fmin(lo.x, c.x), fmin(lo.y, c.y), fmin(lo.z, c.z)};
      hi = d3{fmax(hi.x, c.x), fmax(hi.y, c.y), fmax(hi.z, c.z)};
    }
    double *o = box + 6 * threadIdx.x;
    o[0] = lo.x, o[1] = lo.y, o[2] = lo.z, o[3] = hi.x, o[4] = hi.y,
    o[5] = hi.z;
  }
  __syncthreads();
  const d3 ilo{box[0], box[1], box[2]}, ihi{box[3], box[4], box[5]};
  const d3 jlo{box[6], box[7], box[8]}, jhi{box[9], box[10], box[11]};
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  for (int64_t k0 = 0; k0 < NS; k0 += 256) {
    const int64_t kk = k0 + (int64_t)threadIdx.x;
    const bool keep =
        kk < NS && (heads[kk / kGroup] >> (kk % kGroup) & 1u) != 0 &&
        may_block_tile(ilo, ihi, jlo, jhi, groups[kk]);
    const uint64_t m = __ballot(keep);
    if (lane == 0) wave_count[wave] = __popcll(m);
    __syncthreads();
    int base = 0, n_cand = 0;
    for (int w = 0; w < 4; ++w) {
      base += w < wave ? wave_count[w] : 0;
      n_cand += wave_count[w];
    }
    if (keep)
      cand[base + __popcll(m & ((1ull << lane) - 1ull))] = (int32_t)kk;
    __syncthreads();
    for (int c = 0; c < n_cand; ++c) {
      if (!__any(alive)) break;
      const int k = __builtin_amdgcn_readfirstlane(cand[c]);
      if (group_blocks(a, b, alive, k, groups[k], recs)) alive = false;
    }
    if (!__syncthreads_or(alive)) break;
  }
  if (valid) vis[i * P + j] = (uint8_t)alive;
}

// Workgroup per query point and 64 patches; its kSightWaves waves share the
// blockers, a run of kGroup at a time, and leave a patch that another wave has
// found blocked.  One or two query points leave most of the chip idle, so the
// length of the walk is what a call waits for: 208 patches as blockers 17 us
// (one thread walking all of them: 221 us), 1,072 21 us (944 us), 6 walls
// 15 us, most of it the kernel's code coming in.
constexpr int kSightWaves = 8;
__global__ __launch_bounds__(64 * kSightWaves) void point_visibility_kernel(
    int64_t NQ, const double *__restrict__ points, int64_t P,
    const double *__restrict__ centers, int64_t NS,
    const BlockerRec *__restrict__ recs,
    const BlockerGroup *__restrict__ groups,
    const uint32_t *__restrict__ heads, uint8_t *__restrict__ vis) {
  __shared__ int32_t blocked[64];
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int64_t q = blockIdx.y;
  const int64_t k = (int64_t)blockIdx.x * 64 + lane;
  if (wave == 0) blocked[lane] = 0;
  __syncthreads();
  bool alive = k < P;
  const d3 a = load3(points + 3 * q);
  d3 b{0, 0, 0};
  if (alive) b = load3(centers + 3 * k);
  const int64_t runs = (NS + kGroup - 1) / kGroup;
  for (int64_t run = wave; run < runs; run += kSightWaves) {
    alive = alive && __hip_atomic_load(blocked + lane, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP) == 0;
    if (!__any(alive)) break;
    for (uint32_t h = heads[run]; h != 0; h &= h - 1) {
      const int64_t s = run * kGroup + __ffs((int)h) - 1;
      if (group_blocks(a, b, alive, s, groups[s], recs)) {
        alive = false;
        __hip_atomic_store(blocked + lane, 1, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }
  __syncthreads();
  if (wave == 0 && k < P) vis[q * P + k] = (uint8_t)(blocked[lane] == 0);
}

// ---------------------------------------------------------------------
// visible-pair list (RadiosityFast.py:377-387), one wave per row i
// ---------------------------------------------------------------------
__global__ __launch_bounds__(256) void visible_pairs_kernel(
    int64_t P, const uint8_t *__restrict__ vis, int64_t *__restrict__ offs,
    int32_t *__restrict__ pairs, int fill) {
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= P) return;
  int64_t pos = fill ? offs[i] : 0;
  for (int64_t base = i + 1; base < P; base += 64) {
    int64_t j = base + lane;
    bool f = j < P && vis[i * P + j] != 0;
    uint64_t m = __ballot(f);
    if (fill && f) {
      uint64_t lt = lane ? (m & ((1ull << lane) - 1ull)) : 0ull;
      int64_t p = pos + __popcll(lt);
      pairs[2 * p] = (int32_t)i;
      pairs[2 * p + 1] = (int32_t)j;
    }
    pos += __popcll(m);
  }
  if (!fill && lane == 0) offs[i] = pos;
}

// ---------------------------------------------------------------------
// universal form factor (universal.py:54-96)
// ---------------------------------------------------------------------

// geometry.py:719-748 _coincidence_check(receiver, source), threshold 1e-6:
// whether any corner of p0 meets any of p1.
__device__ inline bool corners_meet(const double *p0, const double *p1, int a,
                                    int b) {
  return norm(load3(p0 + 3 * a) - load3(p1 + 3 * b)) < 1e-6;
}
__device__ inline bool coincident(const double *p0, const double *p1) {
  for (int a = 0; a < 4; ++a)
    for (int b = 0; b < 4; ++b)
      if (corners_meet(p0, p1, a, b)) return true;
  return false;
}

// integration.py:608-651 _sample_boundary_regular, point q of a 4-corner
// patch sampled with n_div segments per side.
__device__ inline d3 boundary_point(const double *el, int q, int n_div) {
  int i = q / n_div, ii = q % n_div;
  d3 a = load3(el + 3 * i), b = load3(el + 3 * ((i + 1) & 3));
  double t = (double)ii, nd = (double)n_div;
  return d3{a.x + (t * (b.x - a.x)) / nd, a.y + (t * (b.y - a.y)) / nd,
            a.z + (t * (b.z - a.z)) / nd};
}

// integration.py:462-486 _newton_cotes_4th (Boole's rule) in its two factors:
// the step's, and the sum over the five values.
__device__ inline double boole_step(double x0, double x1) {
  return (2.0 * (x1 - x0)) / 45.0;
}
__device__ inline double boole_sum(const double *y) {
  return (((7.0 * y[0] + 32.0 * y[1]) + 12.0 * y[2]) + 32.0 * y[3]) +
         7.0 * y[4];
}

// What the lanes of one wave write to LDS before is read after.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// integration.py:38-114 stokes_integration, two pairs per wavefront (eight
// per workgroup: one pair per workgroup is bound by how fast workgroups
// start), a half of the wave for each where a pair has no more than 32 values
// to form.  Whatever several terms share is formed once, by one lane each:
// the 2x16 boundary points, the step factor of each segment and coordinate
// (NaN where the reference skips the segment), Boole's sum over the 16x16
// ln|r| table, which is the same for the three coordinates.  One lane only
// adds the twelve outer terms, in the reference's (dim, segment) order.
// Bound by the float64 logarithms and square roots of the table: 7.4 M pairs
// of a canyon in 9.0 ms; one pair per wavefront 9.8; with 48 lanes forming
// each segment's nodes anew and one all outer terms 21.
constexpr int kStokesPairs = 2;  // of a wave

__global__ __launch_bounds__(256) void stokes_kernel(
    int64_t P, const double *__restrict__ pts, const double *__restrict__ areas,
    int64_t V, const int32_t *__restrict__ pairs, double *__restrict__ ff) {
  constexpr double kSkip = __builtin_nan("");
  struct Pair {
    double point[2][3][16];  // patch i's and j's boundary points, by dim
    double step[2][3][4];
    double form[16][17];
    double sum[16][4];
    double inner[3][16];
    double outer[12];
  };
  __shared__ Pair sh[4 * kStokesPairs];
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  const int half = lane >> 5, l = lane & 31;
  const int64_t v = ((int64_t)blockIdx.x * 4 + wave) * kStokesPairs + half;
  Pair *const two = sh + wave * kStokesPairs;
  Pair &own = two[half];  // this half's pair
  int64_t i = -1, j = -1;
  if (v < V) i = pairs[2 * v], j = pairs[2 * v + 1];
  bool ok = i >= 0 && j >= 0 && i < P && j < P;  // else an invalid pair: skip
  const double *pi = pts + (ok ? 12 * i : 0), *pj = pts + (ok ? 12 * j : 0);
  // coincident pairs are nusselt_kernel's
  const uint64_t meet = __ballot(l < 16 && corners_meet(pj, pi, l >> 2, l & 3));
  ok = ok && (uint32_t)(meet >> (32 * half)) == 0;
  const uint64_t live = __ballot(ok);
  if (live == 0) return;  // uniform; no workgroup barrier follows
  if (ok) {
    const d3 p = boundary_point(l < 16 ? pi : pj, l & 15, 4);
    double(*o)[16] = own.point[l >> 4];
    o[0][l & 15] = p.x, o[1][l & 15] = p.y, o[2][l & 15] = p.z;
  }
  wave_lds_sync();
  if (ok && l < 24) {
    const int dim = (l % 12) >> 2, s = l & 3;
    const double *x = own.point[l / 12][dim];
    const bool take = fabs(x[(4 * s + 4) & 15] - x[4 * s]) > 1e-3;
    own.step[l / 12][dim][s] =
        take ? boole_step(x[4 * s], x[4 * s + 1]) : kSkip;
  }
  double y[5];
  for (int h = 0; h < kStokesPairs; ++h) {
    if ((live >> (32 * h) & 1) == 0) continue;  // uniform
    Pair &w = two[h];
    const int q = lane & 15;
    const d3 b{w.point[1][0][q], w.point[1][1][q], w.point[1][2][q]};
    for (int a = lane >> 4; a < 16; a += 4)
      w.form[a][q] = log(norm(
          d3{w.point[0][0][a], w.point[0][1][a], w.point[0][2][a]} - b));
  }
  wave_lds_sync();
  for (int h = 0; h < kStokesPairs; ++h) {
    Pair &w = two[h];
    const int a = lane >> 2, s = lane & 3;
    for (int k = 0; k < 5; ++k) y[k] = w.form[a][(4 * s + k) & 15];
    w.sum[a][s] = boole_sum(y);
  }
  wave_lds_sync();
  for (int t = lane; t < 48 * kStokesPairs; t += 64) {
    Pair &w = two[t / 48];
    const int a = t % 48 / 3, dim = t % 3;
    double acc = 0.0;
    for (int s = 0; s < 4; ++s) {
      const double h = w.step[1][dim][s];
      if (h == h) acc += h * w.sum[a][s];
    }
    w.inner[dim][a] = acc;
  }
  wave_lds_sync();
  if (ok && l < 12) {
    const int dim = l >> 2, s = l & 3;
    const double h = own.step[0][dim][s];
    for (int k = 0; k < 5; ++k) y[k] = own.inner[dim][(4 * s + k) & 15];
    own.outer[l] = h == h ? h * boole_sum(y) : 0.0;
  }
  wave_lds_sync();
  if (ok && l == 0) {
    double outer = 0.0;
    for (int t = 0; t < 12; ++t) outer += own.outer[t];
    ff[i * P + j] = fabs(outer / ((2.0 * M_PI) * areas[i]));
  }
}

// 3x3 inverse by elimination with partial pivoting, column-wise solve of
// A X = I (np.linalg.inv's LU route).
__device__ inline void inv3(const double (&a_in)[3][3], double (&out)[3][3]) {
  double a[3][3];
  int piv[3] = {0, 1, 2};
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) a[r][c] = a_in[r][c];
  for (int k = 0; k < 3; ++k) {
    int p = k;
    double best = fabs(a[k][k]);
    for (int r = k + 1; r < 3; ++r)
      if (fabs(a[r][k]) > best) {
        best = fabs(a[r][k]);
        p = r;
      }
    if (p != k) {
      for (int c = 0; c < 3; ++c) {
        double t = a[k][c];
        a[k][c] = a[p][c];
        a[p][c] = t;
      }
      int t = piv[k];
      piv[k] = piv[p];
      piv[p] = t;
    }
    for (int r = k + 1; r < 3; ++r) {
      a[r][k] = a[r][k] / a[k][k];
      for (int c = k + 1; c < 3; ++c) a[r][c] = a[r][c] - a[r][k] * a[k][c];
    }
  }
  for (int col = 0; col < 3; ++col) {
    double y[3];
    for (int r = 0; r < 3; ++r) {
      double s = (piv[r] == col) ? 1.0 : 0.0;
      for (int c = 0; c < r; ++c) s = s - a[r][c] * y[c];
      y[r] = s;
    }
    for (int r = 2; r >= 0; --r) {
      double s = y[r];
      for (int c = r + 1; c < 3; ++c) s = s - a[r][c] * out[c][col];
      out[r][col] = s / a[r][r];
    }
  }
}

// integration.py:416-460 _area_under_curve (order 2) with
// _poly_estimation_Lagrange (:349-382) and _poly_integration (:385-412).
__device__ inline double area_under_curve(d2 p0, d2 p1, d2 p2) {
  d2 f = p2 - p0;
  double nf = norm(f);
  d2 r0{f.x / nf, f.y / nf};
  d2 r1{-f.y / nf, f.x / nf};
  double x[3] = {0.0, 0.0, 0.0}, y[3] = {0.0, 0.0, 0.0};
  d2 c1 = p1 - p0, c2 = p2 - p0;
  x[1] = dot(r0, c1);
  y[1] = dot(r1, c1);
  x[2] = dot(r0, c2);
  y[2] = dot(r1, c2);
  double co[3];
  if (fabs(x[2] - x[0]) < 1e-6) {
    co[0] = co[1] = co[2] = 0.0;
  } else {
    double xm[3][3], inv[3][3];
    for (int r = 0; r < 3; ++r)
      for (int o = 0; o < 3; ++o) xm[r][2 - o] = pow(x[r], (double)o);
    inv3(xm, inv);
    for (int r = 0; r < 3; ++r)
      co[r] = (inv[r][0] * y[0] + inv[r][1] * y[1]) + inv[r][2] * y[2];
  }
  double out = 0.0;
  for (int r = 0; r < 3; ++r) {
    double p = (double)(3 - r);
    out += (co[r] * pow(x[2], p)) / p;
    out -= (co[r] * pow(x[0], p)) / p;
  }
  return out;
}

__device__ inline d2 project2(const double *m0, const double *m1, d3 v) {
  return d2{dot(load3(m0), v), dot(load3(m1), v)};
}

// integration.py:116-230 nusselt_analog
__device__ double nusselt_analog(d3 origin, const double *m0,
                                 const double *m1, const double *pj,
                                 const double *nj) {
  d3 sph[8];
  d2 pln[8];
  for (int q = 0; q < 8; ++q) {
    d3 d = boundary_point(pj, q, 2) - origin;
    sph[q] = div(d, norm(d));
    pln[q] = project2(m0, m1, sph[q]);
  }
  d3 e1 = load3(pj + 3) - load3(pj), e2 = load3(pj + 6) - load3(pj + 3);
  double hand = sgn(dot(cross(e1, e2), load3(nj)));
  // _polygon_area of the projected corners (samples 0, 2, 4, 6; z = 0)
  double big_poly = 0.0;
  {
    d3 q0{pln[0].x, pln[0].y, 0.0};
    for (int t = 0; t < 2; ++t) {
      d3 qa{pln[2 * (t + 1)].x, pln[2 * (t + 1)].y, 0.0};
      d3 qb{pln[2 * (t + 2)].x, pln[2 * (t + 2)].y, 0.0};
      big_poly += 0.5 * norm(cross(qa - q0, qb - q0));
    }
  }
  double curved = 0.0;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    int s0 = 2 * jj, s1 = 2 * jj + 1, s2 = (2 * jj + 2) & 7;
    d3 pa{pln[s2].x, pln[s2].y, 0.0}, pb{pln[s0].x, pln[s0].y, 0.0};
    if (!(norm(cross(pa, pb)) > 1e-6)) continue;
    if (dot(pln[s2], pln[s0]) >= 1e-6) {
      curved += area_under_curve(pln[s0], pln[s1], pln[s2]);
    } else {
      d3 mpoint{sph[s0].x + (sph[s2].x - sph[s0].x) / 2.0,
                sph[s0].y + (sph[s2].y - sph[s0].y) / 2.0,
                sph[s0].z + (sph[s2].z - sph[s0].z) / 2.0};
      d3 marc = div(mpoint, norm(mpoint));
      d3 a{sph[s0].x + (marc.x - sph[s0].x) / 2.0,
           sph[s0].y + (marc.y - sph[s0].y) / 2.0,
           sph[s0].z + (marc.z - sph[s0].z) / 2.0};
      d3 b{marc.x + (sph[s2].x - marc.x) / 2.0,
           marc.y + (sph[s2].y - marc.y) / 2.0,
           marc.z + (sph[s2].z - marc.z) / 2.0};
      d2 mp2 = project2(m0, m1, mpoint);
      d2 marc2 = project2(m0, m1, marc);
      d2 a2 = project2(m0, m1, div(a, norm(a)));
      d2 b2 = project2(m0, m1, div(b, norm(b)));
      double lin = (norm(pln[s2] - pln[s0]) * norm(mp2 - marc2)) / 2.0;
      double left = area_under_curve(pln[s0], a2, marc2);
      double right = area_under_curve(marc2, b2, pln[s2]);
      curved += ((lin * sgn(left)) + left) + right;
    }
  }
  return big_poly + hand * curved;
}

// numpy.linspace(0, stop, num)[k]
__device__ inline double linspace0(double stop, int num, int k) {
  if (num == 1) return 0.0;
  if (k == num - 1) return stop;
  return (double)k * (stop / (double)(num - 1)) + 0.0;
}

// integration.py:232-289 nusselt_integration over the regular grid of
// integration.py:533-605 for the pairs that share a corner.  Each lane (of
// the first per_wave) looks at one pair; the wavefront then takes the pairs found, one after the other,
// with one lane per sample and the samples summed in the reference's order by
// lane 0.  A pair in a few hundred shares a corner, so a wavefront for each
// pair is bound by starting them: 7.4 M pairs of a canyon in 0.6 ms instead
// of 9.7 ms.
__global__ __launch_bounds__(64) void nusselt_kernel(
    int64_t P, const double *__restrict__ pts,
    const double *__restrict__ normals, int64_t V, int per_wave,
    const int32_t *__restrict__ pairs, double *__restrict__ ff) {
  __shared__ double vals[64];
  __shared__ double m[6];
  const int lane = threadIdx.x;
  int64_t i = -1, j = -1;
  {
    const int64_t v = (int64_t)blockIdx.x * per_wave + lane;
    if (lane < per_wave && v < V) i = pairs[2 * v], j = pairs[2 * v + 1];
  }
  uint64_t found =
      __ballot(i >= 0 && j >= 0 && i < P && j < P &&
               coincident(pts + 12 * j, pts + 12 * i));
  for (; found != 0; found &= found - 1) {
    const int from = __ffsll((unsigned long long)found) - 1;
    const int64_t fi = __shfl((int)i, from), fj = __shfl((int)j, from);
    const double *pi = pts + 12 * fi, *pj = pts + 12 * fj;
    if (lane == 0) rotation_rows(normals + 3 * fi, m, m + 3);
    d3 u = load3(pi + 3) - load3(pi), w = load3(pi + 9) - load3(pi);
    double nu = norm(u), nw = norm(w);
    double sq = sqrt(1.0 * 64.0);
    int npx = (int)rint(nu / nw * sq);
    int npz = (int)rint(nw / nu * sq);
    if (npz == 0) npz = 1;
    if (npx == 0) npx = 1;
    const int n = npx * npz;
    const double stx = 1.0 - 1.0 / (double)npx, stz = 1.0 - 1.0 / (double)npz;
    const double ssx = 1.0 / (double)(npx * 2), ssz = 1.0 / (double)(npz * 2);
    __syncthreads();
    double out = 0.0;
    for (int base = 0; base < n; base += 64) {
      int q = base + lane;
      if (q < n) {
        int a = q / npz, b = q % npz;
        double s = linspace0(stx, npx, a) + ssx;
        double t = linspace0(stz, npz, b) + ssz;
        d3 p0{(s * u.x + t * w.x) + pi[0], (s * u.y + t * w.y) + pi[1],
              (s * u.z + t * w.z) + pi[2]};
        vals[lane] = nusselt_analog(p0, m, m + 3, pj, normals + 3 * fj);
      }
      __syncthreads();
      if (lane == 0) {
        int cnt = n - base < 64 ? n - base : 64;
        for (int k = 0; k < cnt; ++k) out += vals[k];
      }
      __syncthreads();
    }
    if (lane == 0) {
      out *= 1.0 / (M_PI * (double)n);
      ff[fi * P + fj] = out;
    }
  }
}

// ---------------------------------------------------------------------
// direction maps
// ---------------------------------------------------------------------
__global__ void direction_map_kernel(int64_t P, const uint8_t *__restrict__ vis,
                                     const double *__restrict__ centers,
                                     int64_t D,
                                     const double *__restrict__ out_dirs,
                                     const int64_t *__restrict__ wall_ids,
                                     int64_t *__restrict__ p2o) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = blockIdx.y;
  if (j >= P) return;
  int64_t r = D;
  if (i != j && (i < j ? vis[i * P + j] : vis[j * P + i])) {
    d3 d = load3(centers + 3 * j) - load3(centers + 3 * i);
    d = div(d, norm(d));
    r = nearest_direction(out_dirs + wall_ids[i] * D * 3, D, d);
  }
  p2o[i * P + j] = r;
}

__global__ void point_direction_kernel(int64_t NQ,
                                       const double *__restrict__ points,
                                       int64_t P,
                                       const double *__restrict__ centers,
                                       int64_t D,
                                       const double *__restrict__ out_dirs,
                                       const int64_t *__restrict__ wall_ids,
                                       int64_t *__restrict__ idx) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t q = blockIdx.y;
  if (k >= P) return;
  d3 d = load3(points + 3 * q) - load3(centers + 3 * k);
  d = div(d, norm(d));
  idx[q * P + k] = nearest_direction(out_dirs + wall_ids[k] * D * 3, D, d);
}

// ---------------------------------------------------------------------
// dense directional form factor (RadiosityFast.py:1234-1272)
// ---------------------------------------------------------------------
__global__ void fft_dense_kernel(int64_t P, const uint8_t *__restrict__ vis,
                                 const double *__restrict__ ff, int64_t B,
                                 const double *__restrict__ centers,
                                 const double *__restrict__ areas,
                                 const double *__restrict__ air,
                                 const int64_t *__restrict__ wall_ids,
                                 int64_t S, int64_t D,
                                 const double *__restrict__ brdf,
                                 const int64_t *__restrict__ brdf_index,
                                 const double *__restrict__ in_dirs,
                                 double *__restrict__ fft) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = blockIdx.y;
  if (j >= P) return;
  double *o = fft + (i * P + j) * D * B;
  bool visible = i != j && (i < j ? vis[i * P + j] : vis[j * P + i]);
  if (!visible) {
    for (int64_t k = 0; k < D * B; ++k) o[k] = 0.0;
    return;
  }
  PairFactor pf = pair_factor(i, j, P, centers, areas, ff, wall_ids, S, D, B,
                              brdf, brdf_index, in_dirs);
  for (int64_t b = 0; b < B; ++b) {
    double ab = air ? exp(-air[b] * pf.distance) : 1.0;
    for (int64_t d = 0; d < D; ++d)
      o[d * B + b] = pair_coef(pf, ab, air != nullptr, d, b, B);
  }
}

// ---------------------------------------------------------------------
// source injection (universal.py:98-147, RadiosityFast.py:988-1034)
// ---------------------------------------------------------------------
__global__ void source_energy_kernel(
    const double *__restrict__ source, int64_t P,
    const double *__restrict__ centers, const double *__restrict__ pts,
    const uint8_t *__restrict__ vis, const double *__restrict__ air,
    int64_t B, const int64_t *__restrict__ wall_ids, int64_t S, int64_t D,
    const double *__restrict__ brdf, const int64_t *__restrict__ brdf_index,
    const double *__restrict__ in_dirs, double *__restrict__ energy0,
    double *__restrict__ e0dir, double *__restrict__ distance) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= P) return;
  const d3 src = load3(source);
  const d3 ck = load3(centers + 3 * k);
  double dist = 0.0, pt = 0.0;
  const bool v = vis[k] != 0;
  if (v) {
    dist = norm(src - ck);
    pt = pt_solution(src, pts + 12 * k, false);
  }
  distance[k] = dist;
  // get_scattering_data_source(source, c_k): nearest incoming direction of
  // wall w_k to unit(source - c_k)
  d3 u = src - ck;
  u = div(u, norm(u));
  const int64_t w = wall_ids[k];
  const int64_t s = nearest_direction(in_dirs + w * S * 3, S, u);
  const double *row = brdf + (brdf_index[w] * S + s) * D * B;
  for (int64_t b = 0; b < B; ++b) {
    double e = 0.0;
    if (v) e = air ? exp(-air[b] * dist) * pt : pt;
    energy0[k * B + b] = e;
    for (int64_t d = 0; d < D; ++d)
      e0dir[(k * D + d) * B + b] = e * row[d * B + b];
  }
}

}  // namespace
}  // namespace spr

using namespace spr;

// Blocker records, groups (at most one per blocker) and group starts.
namespace {
struct Blockers {
  const BlockerRec *recs;
  const BlockerGroup *groups;
  const uint32_t *heads;
};
}  // namespace

extern "C" int64_t spr_visibility_workspace(int64_t NS) {
  if (NS < 0) return -1;
  const int64_t n = NS > 0 ? NS : 1;
  return (int64_t)(sizeof(BlockerRec) + sizeof(BlockerGroup)) * n +
         (int64_t)sizeof(uint32_t) * ceil_div(n, kGroup);
}

static int build_blockers(int64_t NS, const double *normals,
                          const double *pts, void *ws, int64_t ws_bytes,
                          hipStream_t s, Blockers &out) {
  if (ws_bytes < spr_visibility_workspace(NS))
    return fail(SPR_ERR_WORKSPACE, "visibility workspace of %lld bytes, "
                "need %lld", (long long)ws_bytes,
                (long long)spr_visibility_workspace(NS));
  auto *recs = static_cast<BlockerRec *>(ws);
  auto *groups = reinterpret_cast<BlockerGroup *>(recs + NS);
  auto *heads = reinterpret_cast<uint32_t *>(groups + NS);
  out = Blockers{recs, groups, heads};
  if (NS == 0) return SPR_OK;
  hipLaunchKernelGGL(blocker_kernel, dim3((unsigned)ceil_div(NS, kGroup)),
                     dim3(4 * kGroup), 0, s, NS, normals, pts, recs, groups, heads);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_p2p_visibility(int64_t P, const double *centers,
                                  int64_t NS, const double *surf_normals,
                                  const double *surf_points, uint8_t *vis,
                                  void *workspace, int64_t workspace_bytes,
                                  void *stream) {
  SPR_REQUIRE(P > 0 && NS >= 0 && P < (int64_t)1 << 20,
              "spr_p2p_visibility: bad sizes");
  SPR_REQUIRE(centers && vis && workspace && (NS == 0 || (surf_normals &&
                                                          surf_points)),
              "spr_p2p_visibility: null pointer");
  hipStream_t s = as_stream(stream);
  Blockers bl;
  int rc = build_blockers(NS, surf_normals, surf_points, workspace,
                          workspace_bytes, s, bl);
  if (rc) return rc;
  unsigned nt = (unsigned)ceil_div(P, 16);
  hipLaunchKernelGGL(p2p_visibility_kernel, dim3(nt, nt), dim3(256), 0, s, P,
                     centers, NS, bl.recs, bl.groups, bl.heads, vis);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_point_visibility(int64_t NQ, const double *points,
                                    int64_t P, const double *centers,
                                    int64_t NS, const double *surf_normals,
                                    const double *surf_points, uint8_t *vis,
                                    void *workspace, int64_t workspace_bytes,
                                    void *stream) {
  SPR_REQUIRE(NQ > 0 && P > 0 && NS >= 0 && NQ < 65536,
              "spr_point_visibility: bad sizes");
  SPR_REQUIRE(points && centers && vis && workspace &&
                  (NS == 0 || (surf_normals && surf_points)),
              "spr_point_visibility: null pointer");
  hipStream_t s = as_stream(stream);
  Blockers bl;
  int rc = build_blockers(NS, surf_normals, surf_points, workspace,
                          workspace_bytes, s, bl);
  if (rc) return rc;
  hipLaunchKernelGGL(point_visibility_kernel,
                     dim3((unsigned)ceil_div(P, 64), (unsigned)NQ),
                     dim3(64 * kSightWaves), 0, s, NQ, points, P, centers, NS,
                     bl.recs, bl.groups, bl.heads, vis);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_visible_pairs(int64_t P, const uint8_t *vis,
                                 int64_t *row_offsets, int32_t *pairs,
                                 void *stream) {
  SPR_REQUIRE(P > 0 && vis && row_offsets, "spr_visible_pairs: bad args");
  hipStream_t s = as_stream(stream);
  unsigned blocks = (unsigned)ceil_div(P, 4);
  if (!pairs) {
    hipLaunchKernelGGL(visible_pairs_kernel, dim3(blocks), dim3(256), 0, s, P,
                       vis, row_offsets, (int32_t *)nullptr, 0);
    SPR_LAUNCH_CHECK();
    return scan_exclusive(row_offsets, P, s);
  }
  hipLaunchKernelGGL(visible_pairs_kernel, dim3(blocks), dim3(256), 0, s, P,
                     vis, row_offsets, pairs, 1);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_form_factors(int64_t P, const double *points,
                                const double *normals, const double *areas,
                                int64_t V, const int32_t *pairs, double *ff,
                                void *stream) {
  SPR_REQUIRE(P > 0 && V >= 0 && V < 0x7fffffff,
              "spr_form_factors: bad sizes");
  SPR_REQUIRE(points && normals && areas && ff && (V == 0 || pairs),
              "spr_form_factors: null pointer");
  hipStream_t s = as_stream(stream);
  int rc = fill<double>(ff, P * P, 0.0, s);
  if (rc || V == 0) return rc;
  hipLaunchKernelGGL(stokes_kernel,
                     dim3((unsigned)ceil_div(V, 4 * kStokesPairs)), dim3(256),
                     0, s, P, points, areas, V, pairs, ff);
  SPR_LAUNCH_CHECK();
  // As few pairs to a wavefront as 16,384 of them allow: in a small scene many
  // pairs share a corner, and those of one wavefront are one after the other.
  int per_wave = 1;
  while (per_wave < 64 && ceil_div(V, per_wave) > 16384) per_wave *= 2;
  hipLaunchKernelGGL(nusselt_kernel, dim3((unsigned)ceil_div(V, per_wave)),
                     dim3(64), 0, s, P, points, normals, V, per_wave, pairs,
                     ff);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_direction_map(int64_t P, const uint8_t *vis,
                                 const double *centers, int64_t D,
                                 const double *out_dirs,
                                 const int64_t *wall_ids, int64_t *p2o,
                                 void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && P < 65536, "spr_direction_map: bad sizes");
  SPR_REQUIRE(vis && centers && out_dirs && wall_ids && p2o,
              "spr_direction_map: null pointer");
  hipLaunchKernelGGL(direction_map_kernel,
                     dim3((unsigned)ceil_div(P, 256), (unsigned)P), dim3(256),
                     0, as_stream(stream), P, vis, centers, D, out_dirs,
                     wall_ids, p2o);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_point_direction_index(int64_t NQ, const double *points,
                                         int64_t P, const double *centers,
                                         int64_t D, const double *out_dirs,
                                         const int64_t *wall_ids,
                                         int64_t *idx, void *stream) {
  SPR_REQUIRE(NQ > 0 && P > 0 && D > 0 && NQ < 65536,
              "spr_point_direction_index: bad sizes");
  SPR_REQUIRE(points && centers && out_dirs && wall_ids && idx,
              "spr_point_direction_index: null pointer");
  hipLaunchKernelGGL(point_direction_kernel,
                     dim3((unsigned)ceil_div(P, 256), (unsigned)NQ),
                     dim3(256), 0, as_stream(stream), NQ, points, P, centers,
                     D, out_dirs, wall_ids, idx);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_fft_dense(int64_t P, const uint8_t *vis, const double *ff,
                             int64_t B, const double *centers,
                             const double *areas, const double *air,
                             const int64_t *wall_ids, int64_t S, int64_t D,
                             const double *brdf, const int64_t *brdf_index,
                             const double *in_dirs, double *fft,
                             void *stream) {
  SPR_REQUIRE(P > 0 && B > 0 && D > 0 && P < 65536,
              "spr_fft_dense: bad sizes");
  SPR_REQUIRE(vis && ff && centers && areas && wall_ids && fft,
              "spr_fft_dense: null pointer");
  SPR_REQUIRE(!brdf || (brdf_index && in_dirs && S > 0),
              "spr_fft_dense: brdf needs brdf_index and in_dirs");
  SPR_REQUIRE(brdf || D == 1, "spr_fft_dense: D must be 1 without a BRDF");
  hipLaunchKernelGGL(fft_dense_kernel,
                     dim3((unsigned)ceil_div(P, 128), (unsigned)P), dim3(128),
                     0, as_stream(stream), P, vis, ff, B, centers, areas, air,
                     wall_ids, S, D, brdf, brdf_index, in_dirs, fft);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_source_energy(const double *source, int64_t P,
                                 const double *centers, const double *points,
                                 const uint8_t *vis, const double *air,
                                 int64_t B, const int64_t *wall_ids,
                                 int64_t S, int64_t D, const double *brdf,
                                 const int64_t *brdf_index,
                                 const double *in_dirs, double *energy0,
                                 double *e0dir, double *distance,
                                 void *stream) {
  SPR_REQUIRE(P > 0 && B > 0 && S > 0 && D > 0,
              "spr_source_energy: bad sizes");
  SPR_REQUIRE(source && centers && points && vis && wall_ids && brdf &&
                  brdf_index && in_dirs && energy0 && e0dir && distance,
              "spr_source_energy: null pointer");
  hipLaunchKernelGGL(source_energy_kernel, dim3((unsigned)ceil_div(P, 128)),
                     dim3(128), 0, as_stream(stream), source, P, centers,
                     points, vis, air, B, wall_ids, S, D, brdf, brdf_index,
                     in_dirs, energy0, e0dir, distance);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}
