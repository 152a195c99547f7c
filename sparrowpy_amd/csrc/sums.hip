// All reflection orders of one source: the order loop, and the sum of the
// orders.
//
// Reference: the order loop of _energy_exchange and its running total
// (sparrowpy/classes/RadiosityFast.py:1073-1145).  With A the exchange of
// one order and E_0 the injected energy (:1037-1070), E_{k+1} = A E_k and the
// result is E_0 + ... + E_K.  Two forms:
//
// spr_exchange_orders carries the order beside the running total (a
// compensated pair of float32): what stepping spr_exchange_gather_* /
// _spread_* does, in one call.  The total starts as the injected energy and
// the last order writes the rounded total alone, so nothing is cleared
// before the loop and no pass follows it.
//
// spr_exchange_sum carries the sum instead of the order, x_{k+1} = E_0 +
// A x_k, x_K being the result: no total to read and write, two state
// buffers instead of four.  It holds fewer bits: the sum is one float32
// rounded every order, where the total above is a pair rounded at the end.
// Its bound is the same, but the error against float64 grows with the orders:
// 94 patches, 10 orders: rms 2.7e-8, as order by order; 200 orders: 4.8e-8
// against 3.0e-8; 6 patches, 200 orders: 7.5e-8 (largest 1.9e-7) against
// 4.5e-8 (1.4e-7).  It runs only where a caller asks for it.
//
// Both run an order only on the bins that energy can have reached: order 0
// ends before bin `reach`, and an order reaches at most the plan's longest
// delay further.  Bins beyond are exact zeros of the reference's loop too;
// they are cleared once, at the end.  In a room the sound crosses in 60 bins
// an order of 2,000 bins is a third of the work on average over 20 orders
// (328 patches, 16 directions, 4 bands: 8.48 -> 5.27 ms when orders took two
// launches; 2.7 with one).  That holds for finite factors only: an infinite or
// NaN one times those zeros is NaN, in the reference's loop from the pair's
// delay on.  Such factors are reported, and the caller runs whole orders.
#include <algorithm>

#include "spr_common.hpp"
#include "spr_exchange.hpp"
#include "spr_util.hpp"

namespace spr {
namespace {

// The factors of a plan: arrays read whole, and of a grouped plan the BRDF
// rows (width values each, 2^lanes threads to a row) of its groups.
struct Factors {
  const double *whole[2] = {};
  int64_t n[2] = {};
  const double *rows = nullptr;
  const int32_t *key = nullptr;
  const int64_t *groups = nullptr;  // how many
  int64_t width = 0;
  int lanes = 0;
};

Factors factors_of(const spr_exchange_plan &p) {
  const int64_t DP = spr_padded_directions(p.D);
  Factors f;
  if (p.kind == SPR_PLAN_PAIRS) {
    f.whole[0] = p.coef, f.n[0] = p.Vd * p.B * DP;
    return f;
  }
  f.whole[0] = p.scal, f.n[0] = p.B * p.Vd;
  if (p.kind == SPR_PLAN_DS) {
    f.whole[1] = p.dscal, f.n[1] = p.B * p.Vd;
  } else {
    f.rows = p.rtab, f.key = p.grp_key, f.groups = p.grp_ptr + p.P;
    f.width = p.B * DP;
    while (f.lanes < 6 && 1 << f.lanes < f.width) ++f.lanes;
  }
  return f;
}

// Bins [t0, t1) of every histogram row: E_0 (with e0dir), or 0; with lo, x
// and lo as a compensated pair and x's rounded value in prev too.  A wave
// takes kFillBins bins of one row at a time; bound by the writes.  The first
// `looks` blocks look over `factors` instead and report infinities and NaN:
// once per call, beside the bins cleared at its end, as a launch of its own
// would wait for loads alone.
constexpr int kFillBins = 1024;

__global__ __launch_bounds__(256) void row_fill_kernel(
    int64_t P, int64_t DB, int64_t T, int64_t t0, int64_t t1, int64_t chunks,
    const double *__restrict__ e0dir, const double *__restrict__ d0, double c,
    double dt, float *__restrict__ x, float *__restrict__ lo,
    float *__restrict__ prev, int32_t *__restrict__ n0, Factors factors,
    uint32_t looks, int *__restrict__ err) {
  const int lane = (int)threadIdx.x & 63;
  if (blockIdx.x < looks) {  // uniform
    bool finite = true;
    const int64_t me = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t threads = 256 * (int64_t)looks;
    for (int a = 0; a < 2; ++a)
#pragma unroll 4
      for (int64_t i = me; i < factors.n[a]; i += threads)
        finite &= fabs(factors.whole[a][i]) < __builtin_inf();
    if (factors.rows) {
      const int64_t n = *factors.groups, w = factors.width;
      const int lanes = factors.lanes;
      for (int64_t g = me >> lanes; g < n; g += threads >> lanes) {
        const double *row = factors.rows + factors.key[g] * w;
        for (int64_t i = me & ((1 << lanes) - 1); i < w; i += 1 << lanes)
          finite &= fabs(row[i]) < __builtin_inf();
      }
    }
    if (!finite) atomicOr(err, 4);
    return;
  }
  const int64_t waves = (int64_t)(gridDim.x - looks) * 4;
  for (int64_t q = (int64_t)(blockIdx.x - looks) * 4 + (threadIdx.x >> 6);
       q < P * DB * chunks; q += waves) {
    const int64_t row = q / chunks, chunk = q % chunks;
    int64_t n = -1;
    float v = 0.f, w = 0.f;
    if (e0dir) {
      const int64_t i = row / DB;
      n = delay_floor(d0[i], c, dt);
      // a delay outside the histogram, or beyond the caller's reach, injects
      // nothing and is reported
      const int bad = n < 0 || n >= T ? 1 : n >= t1 ? 2 : 0;
      if (bad) n = -1;
      if (chunk == 0 && lane == 0 && row % DB == 0) {
        n0[i] = (int32_t)n;
        if (bad) atomicOr(err, bad);
      }
      const double e = e0dir[row];
      v = (float)e;
      w = (float)(e - (double)v);
    }
    const int64_t a = t0 + chunk * kFillBins;
    const int64_t b = a + kFillBins < t1 ? a + kFillBins : t1;
    for (int64_t t = a + lane; t < b; t += 64) {
      x[row * T + t] = t == n ? v : 0.f;
      if (lo) {
        lo[row * T + t] = t == n ? w : 0.f;
        prev[row * T + t] = t == n ? v : 0.f;
      }
    }
  }
}

int fill_rows(const spr_exchange_plan &p, int64_t T, int64_t t0, int64_t t1,
              const double *e0dir, const double *d0, double c, double dt,
              float *x, float *lo, float *prev, int32_t *n0, int *err,
              hipStream_t s, bool look = false) {
  const Factors factors = look ? factors_of(p) : Factors{};
  // 2 values or rows to a thread, as far as 2,048 blocks go
  const int64_t values = std::max(
      factors.n[0], factors.rows ? p.P * p.max_groups << factors.lanes : 0);
  const int64_t looks =
      look ? std::min<int64_t>(ceil_div(values, 512), 2048) : 0;
  const int64_t chunks = t1 > t0 ? ceil_div(t1 - t0, kFillBins) : 0;
  const int64_t nb = ceil_div(p.P * p.D * p.B * chunks, 4);
  if (!looks && !nb) return SPR_OK;
  hipLaunchKernelGGL(row_fill_kernel,
                     dim3((unsigned)(looks + std::min<int64_t>(nb, 1 << 20))),
                     dim3(256), 0, s, p.P, p.D * p.B, T, t0, t1, chunks,
                     e0dir, d0, c, dt, x, lo, prev, n0, factors,
                     (uint32_t)looks, err);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

int check_plan(const char *name, const spr_exchange_plan &p) {
  SPR_REQUIRE(p.row_ptr && p.lag, "%s: null plan array", name);
  if (p.kind == SPR_PLAN_PAIRS) {
    SPR_REQUIRE(p.src && p.dir && p.coef, "%s: null plan array", name);
    return SPR_OK;
  }
  SPR_REQUIRE(p.kind == SPR_PLAN_GROUPED || p.kind == SPR_PLAN_DS,
              "%s: unknown plan kind %lld", name, (long long)p.kind);
  SPR_REQUIRE(p.grp_ptr && p.grp_key && p.rowid && p.scal,
              "%s: null plan array", name);
  // (without grp_start a grouped plan's keys are its groups' first entries;
  // a diffuse + specular plan's keys are directions)
  SPR_REQUIRE(p.kind == SPR_PLAN_DS ? p.dscal && p.grp_start
                                    : p.rtab != nullptr,
              "%s: null plan array", name);
  SPR_REQUIRE(p.max_groups > 0, "%s: max_groups must be positive", name);
  if (!p.M) return SPR_OK;
  SPR_REQUIRE(p.tile_slots > 0 && p.tptr && p.gstart && p.mlag && p.mw,
              "%s: null tile array", name);
  if (p.kind == SPR_PLAN_DS)
    SPR_REQUIRE(p.tile_rows == 16 && p.gdiff && p.mspan && p.mdw,
                "%s: diffuse + specular tiles have 16 rows", name);
  else if (p.tile_rows == 16)
    SPR_REQUIRE(p.mspan && (p.tile_r == 8 || p.tile_r == 16),
                "%s: 16-row tiles gather 8 or 16 bins per lane", name);
  else
    SPR_REQUIRE(p.mrow && (p.tile_rows == 4 || p.tile_rows == 8),
                "%s: tiles have 4, 8 or 16 rows", name);
  return SPR_OK;
}

// The arguments both forms share; *K becomes 0 where there is no order to
// run (none asked for, or no pair of patches sees another).
int check_call(const char *name, const spr_exchange_plan &p, int64_t T,
               int64_t *K, int64_t reach, const double *e0dir,
               const double *d0, double c, double dt, const float *out, const float *gsum,
               const int32_t *n0, const int *err_flag) {
  SPR_REQUIRE(p.P > 0 && p.D > 0 && p.B > 0 && p.Vd >= 0 && T > 0 && c > 0 &&
                  dt > 0,
              "%s: bad sizes", name);
  SPR_REQUIRE(e0dir && d0 && out && n0 && err_flag, "%s: null pointer", name);
  SPR_REQUIRE(reach > 0 && p.max_lag >= 0, "%s: bad reach", name);
  if (*K < 0 || p.Vd == 0) *K = 0;
  if (!*K) return SPR_OK;
  SPR_REQUIRE(T < 0x3fffffff, "%s: histogram too long", name);
  SPR_REQUIRE(spr_padded_directions(p.D) > 0,
              "%s: D=%lld unsupported (max 64)", name, (long long)p.D);
  SPR_REQUIRE(p.kind == SPR_PLAN_PAIRS || gsum, "%s: null pointer", name);
  return check_plan(name, p);
}

// One order of a grouped or diffuse + specular plan: y = A x (plus the
// step's injection), the total updated with it and with `pair`.  gsum is
// left with the group sums if keep is set (with y null: only they are formed).
int order(const spr_exchange_plan &p, int64_t T, const float *x,
          const float *pair, float *y, float *hi, float *lo, float *gsum,
          bool keep, const OrderStep &step, hipStream_t s) {
  if (const int R = row_shape(p, T, step.span))
    return row_order(p, R, T, x, pair, y, hi, lo, keep ? gsum : nullptr, step,
                     s);
  const int rc = p.M ? gather_tiles(p, T, x, gsum, step, s)
                     : gather_rows(p, T, x, gsum, step, s);
  return rc || !y ? rc : spread_rows(p, T, gsum, pair, y, hi, lo, step, s);
}

// Bins that order k can hold energy in.
int64_t reached(const spr_exchange_plan &p, int64_t T, int64_t reach,
                int64_t k) {
  return std::min(T, std::min(T, reach) + k * std::min(T, p.max_lag));
}

// The step from order k to k + 1, without a total.
OrderStep step_from(const spr_exchange_plan &p, int64_t T, int64_t reach,
                    int64_t k) {
  return {{(int)reached(p, T, reach, k), (int)reached(p, T, reach, k + 1), 0, 0,
           0},
          {}};
}

// What both backward segments check; recomputes orders k0 + 1 .. k0 + n - 1
// from states[0] = E_k0, gsums (if not null) receiving the group sums of the
// orders k0 .. k0 + n - 2.
int recompute(const char *name, const spr_exchange_plan *plan, int64_t kind,
              int64_t T, int64_t k0, int64_t n, int64_t reach,
              float *const *states, float *gsum, float *const *gsums,
              hipStream_t s) {
  SPR_REQUIRE(plan && plan->kind == kind, "%s: bad plan", name);
  const spr_exchange_plan &p = *plan;
  SPR_REQUIRE(p.P > 0 && p.P < ((int64_t)1 << 25) && p.D > 0 && p.D <= 64 &&
                  p.B > 0 && p.Vd > 0 && T > 0 && T < ((int64_t)1 << 29) &&
                  k0 >= 0 && n > 0 && reach > 0 && p.max_lag >= 0,
              "%s: bad sizes", name);
  int rc = check_plan(name, p);
  if (rc) return rc;
  for (int64_t i = 0; i < n; ++i)
    SPR_REQUIRE(states[i] && (!gsums || gsums[i]), "%s: null pointer", name);
  for (int64_t i = 0; i + 1 < n; ++i)
    if ((rc = order(p, T, states[i], nullptr, states[i + 1], nullptr, nullptr,
                    gsums ? gsums[i] : gsum, gsums != nullptr,
                    step_from(p, T, reach, k0 + i), s)))
      return rc;
  return SPR_OK;
}

}  // namespace
}  // namespace spr

using namespace spr;

extern "C" int spr_exchange_sum(const spr_exchange_plan *plan, int64_t T,
                                int64_t K, int64_t reach,
                                const double *e0dir, const double *d0,
                                double c, double dt,
                                float *out, float *tmp, float *gsum,
                                int32_t *n0, int *err_flag, void *stream) {
  SPR_REQUIRE(plan, "spr_exchange_sum: null plan");
  const spr_exchange_plan &p = *plan;
  int rc = check_call("spr_exchange_sum", p, T, &K, reach, e0dir, d0, c, dt, out,
                      gsum, n0, err_flag);
  if (rc) return rc;
  SPR_REQUIRE(!K || (tmp && tmp != out), "spr_exchange_sum: null pointer");
  hipStream_t s = as_stream(stream);
  float *x = K % 2 ? tmp : out, *y = K % 2 ? out : tmp;
  int64_t Tc = K ? std::min(T, reach) : T;
  if ((rc = fill_rows(p, T, 0, Tc, e0dir, d0, c, dt, x, nullptr, nullptr, n0,
                      err_flag, s)))
    return rc;
  const bool limited = Tc < T;
  OrderStep step{{0, 0, 0, 0, 0}, {e0dir, n0}};
  for (int64_t k = 0; k < K; ++k) {
    step.span.Tp = (int)Tc;
    step.span.Tc = (int)(Tc = std::min(T, Tc + p.max_lag));
    if (p.kind == SPR_PLAN_PAIRS) {
      rc = step_pairs(p.P, p.D, p.B, T, p.row_ptr, p.src, p.lag, p.dir,
                      p.coef, x, y, nullptr, nullptr, &step, s);
    } else {
      rc = order(p, T, x, nullptr, y, nullptr, nullptr, gsum, false, step, s);
    }
    if (rc) return rc;
    std::swap(x, y);
  }
  return fill_rows(p, T, Tc, T, nullptr, nullptr, c, dt, out, nullptr, nullptr,
                   nullptr, err_flag, s, limited);
}

int spr::exchange_orders(const char *name, const spr_exchange_plan &p,
                         int64_t T, int64_t K, int64_t reach,
                         const double *e0dir, const double *d0, double c,
                         double dt, float *out, float *lo,
                         float *const *states, int64_t n_states, float *gsum,
                         int32_t *n0, int *err_flag, hipStream_t s) {
  int rc = check_call(name, p, T, &K, reach, e0dir, d0, c, dt, out, gsum, n0,
                      err_flag);
  if (rc) return rc;
  SPR_REQUIRE(!K || (lo && states), "%s: null pointer", name);
  for (int64_t k = 0; k < std::min(K, n_states); ++k)
    SPR_REQUIRE(states[k] && (k == 0 || states[k] != states[k - 1]),
                "%s: orders need a buffer each, two in turn at least", name);
  int64_t Tc = K ? std::min(T, reach) : T;
  if ((rc = fill_rows(p, T, 0, Tc, e0dir, d0, c, dt, out, K ? lo : nullptr,
                      K ? states[0] : nullptr, n0, err_flag, s)))
    return rc;
  const bool limited = Tc < T;
  OrderStep step{{0, 0, (int)Tc, 0, 0}, {}};
  OrderSpan &sp = step.span;
  for (int64_t k = 1; k <= K; ++k) {
    sp.Tp = (int)Tc;
    sp.Tc = (int)(Tc = std::min(T, Tc + p.max_lag));
    sp.last = k == K;
    const float *prev = states[(k - 1) % n_states];
    // (the last order is not stored)
    float *cur = sp.last ? lo : states[k % n_states];
    bool add = true;
    if (p.kind == SPR_PLAN_PAIRS) {
      rc = step_pairs(p.P, p.D, p.B, T, p.row_ptr, p.src, p.lag, p.dir,
                      p.coef, prev, cur, out, lo, &step, s);
    } else {
      // the total takes two orders at a time (the even ones' spread); an
      // odd last order is added on its own, as rounded
      const bool pair = k % 2 == 0;
      add = pair || sp.last;
      sp.round = add && !pair;
      rc = order(p, T, prev, pair ? prev : nullptr, cur, add ? out : nullptr,
                 add ? lo : nullptr, gsum, false, step, s);
    }
    if (rc) return rc;
    if (add) sp.Tv = sp.Tc;
  }
  return fill_rows(p, T, Tc, T, nullptr, nullptr, c, dt, out, nullptr, nullptr,
                   nullptr, err_flag, s, limited);
}

extern "C" int spr_exchange_orders(const spr_exchange_plan *plan, int64_t T,
                                   int64_t K, int64_t reach,
                                   const double *e0dir, const double *d0,
                                   double c, double dt, float *out, float *lo,
                                   float *const *states, float *gsum,
                                   int32_t *n0, int *err_flag, void *stream) {
  SPR_REQUIRE(plan, "spr_exchange_orders: null plan");
  return exchange_orders("spr_exchange_orders", *plan, T, K, reach, e0dir, d0,
                         c, dt, out, lo, states, std::max<int64_t>(K, 1), gsum,
                         n0, err_flag, as_stream(stream));
}

extern "C" int spr_adjoint_segment_ds(
    const spr_exchange_plan *plan, int64_t T, int64_t k0, int64_t n,
    int64_t reach, float *const *states, float *gsum, const int64_t *tgptr,
    const int32_t *tkey, const int32_t *tlag, const int32_t *tm,
    const double *twa, const double *twc, const float *lam,
    const float *mu_next, float *mu_even, float *mu_odd, float *musum,
    double *ga, void *stream) {
  SPR_REQUIRE(states && gsum && tgptr && tkey && tlag && tm && twa && twc &&
                  lam && mu_next && mu_even && mu_odd && musum && ga,
              "spr_adjoint_segment_ds: null pointer");
  hipStream_t s = as_stream(stream);
  int rc = recompute("spr_adjoint_segment_ds", plan, SPR_PLAN_DS, T, k0, n,
                     reach, states, gsum, nullptr, s);
  if (rc) return rc;
  const spr_exchange_plan &p = *plan;
  const float *mu = mu_next;
  for (int64_t k = k0 + n - 1; k >= k0; --k) {
    const int64_t Tk = reached(p, T, reach, k);
    const int64_t Tn = reached(p, T, reach, k + 1);
    float *out = k % 2 ? mu_odd : mu_even;
    SPR_REQUIRE(out != mu && out != lam, "spr_adjoint_segment_ds: aliased mu");
    if ((rc = direction_sum(p.P, p.D, p.B, T, Tn, mu, musum, s))) return rc;
    if ((rc = adjoint_ds(p.P, p.D, p.B, T, Tk, Tn, p.Vd, tgptr, tkey, tlag, tm,
                         twa, twc, lam, musum, mu, states[k - k0], out, ga,
                         s)))
      return rc;
    mu = out;
  }
  return SPR_OK;
}

extern "C" int spr_adjoint_segment_grouped(
    const spr_exchange_plan *plan, int64_t T, int64_t k0, int64_t n,
    int64_t reach, float *const *states, float *const *gsums,
    const int64_t *trow_ptr, const int32_t *tgrp, const int32_t *tlag,
    const double *tscal, const float *lam, const float *mu_next,
    float *mu_even, float *mu_odd, float *nu, double *gg, void *stream) {
  SPR_REQUIRE(states && gsums && trow_ptr && tgrp && tlag && tscal && lam &&
                  mu_next && mu_even && mu_odd && nu && gg,
              "spr_adjoint_segment_grouped: null pointer");
  hipStream_t s = as_stream(stream);
  int rc = recompute("spr_adjoint_segment_grouped", plan, SPR_PLAN_GROUPED, T,
                     k0, n, reach, states, nullptr, gsums, s);
  if (rc) return rc;
  const spr_exchange_plan &p = *plan;
  const float *mu = mu_next;
  for (int64_t k = k0 + n - 1; k >= k0; --k) {
    const int64_t i = k - k0;
    const int64_t Tk = reached(p, T, reach, k);
    const int64_t Tn = reached(p, T, reach, k + 1);
    float *out = k % 2 ? mu_odd : mu_even;
    SPR_REQUIRE(out != mu && out != lam,
                "spr_adjoint_segment_grouped: aliased mu");
    // the last order's group sums are still to be formed, and those whose
    // buffer a later order took
    if ((i == n - 1 || gsums[i] == gsums[n - 1]) &&
        (rc = order(p, T, states[i], nullptr, nullptr, nullptr, nullptr,
                    gsums[i], true, step_from(p, T, reach, k), s)))
      return rc;
    if ((rc = table_grad(p.P, p.D, p.B, T, Tn, p.grp_ptr, mu, gsums[i], gg,
                         s)))
      return rc;
    if ((rc = spread_adjoint(p.P, p.D, p.B, T, Tn, p.grp_ptr, p.grp_key,
                             p.rtab, mu, nu, s)))
      return rc;
    if ((rc = gather_adjoint(p.P, p.D, p.B, T, Tk, Tn, p.Vd, trow_ptr, tgrp,
                             tlag, tscal, nu, lam, out, s)))
      return rc;
    mu = out;
  }
  return SPR_OK;
}
