// Adjoint of the energy exchange on a diffuse + specular plan.
//
// Forward (RadiosityFast.py:1073-1145): E_{k+1}[j,d,b,t] = sum over entries
// e = (i -> j) of F~_e[d,b] * E_k[i, dir_e, b, t - n_e], total = sum_k E_k,
// with F~_e[d,b] = w_eb (A[k_e,b] + C[k_e,b] [d = m_e]) (A: diffuse
// constant, C: specular part of BRDF row k_e; w_eb the pair factor).
// For a loss L(total) with lambda = dL/dtotal:
//   mu_K = lambda,  mu_k = lambda + A^T mu_{k+1},
//   (A^T mu)[i,d',b,t] = sum_{e: i -> j, dir_e = d'}
//        w_eb (A_b sum_d mu[j,d,b,t+n_e] + C_b mu[j,m_e,b,t+n_e]),
//   dL/d(w A)_eb += sum_t (sum_d mu_{k+1}[j,d,b,t]) E_k[i,d',b,t-n_e],
//   dL/d(w C)_eb += sum_t mu_{k+1}[j,m_e,b,t] E_k[i,d',b,t-n_e],
// and dL/dE_0 = mu_0, which reaches the tables through the injection
// E_0dir[i,:,b] = E0[i,b] (A + C e_m)[k0_i, b] (RadiosityFast.py:988-1034).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "spr_common.hpp"
#include "spr_exchange.hpp"
#include "spr_util.hpp"

namespace spr {
namespace {

// scal[b,e] = wgt[b,e] C[krow_e, b], dscal[b,e] = wgt[b,e] A[krow_e, b]
__global__ void ds_weights_kernel(int64_t B, int64_t Vd,
                                  const int32_t *__restrict__ krow,
                                  const double *__restrict__ wgt,
                                  const double *__restrict__ ta,
                                  const double *__restrict__ tc,
                                  double *__restrict__ scal,
                                  double *__restrict__ dscal) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= B * Vd) return;
  const int64_t b = q / Vd, e = q % Vd;
  const int64_t k = krow[e];
  scal[q] = wgt[q] * tc[k * B + b];
  dscal[q] = wgt[q] * ta[k * B + b];
}

// Transposed weights: twa[b,q] = dscal[b, te[q]], twc[b,q] = scal[b, te[q]].
__global__ void t_weights_kernel(int64_t B, int64_t Vd,
                                 const int32_t *__restrict__ te,
                                 const double *__restrict__ scal,
                                 const double *__restrict__ dscal,
                                 double *__restrict__ twa,
                                 double *__restrict__ twc) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= B * Vd) return;
  const int64_t b = q / Vd, p = q % Vd;
  const int64_t e = te[p];
  twa[q] = dscal[b * Vd + e];
  twc[q] = scal[b * Vd + e];
}

// Injection from the tables: k0[p] = BRDF row of patch p for the direction
// of the source, e0dir[p,d,b] = energy0[p,b] (A[k0,b] + C[k0,b] [d = m]).
__global__ void ds_injection_kernel(
    int64_t P, int64_t D, int64_t B, const double *__restrict__ source,
    const double *__restrict__ centers, const int64_t *__restrict__ wall_ids,
    int64_t S, const int64_t *__restrict__ brdf_index,
    const double *__restrict__ in_dirs, const double *__restrict__ energy0,
    const double *__restrict__ ta, const double *__restrict__ tc,
    const int32_t *__restrict__ spec_dir, int32_t *__restrict__ k0,
    double *__restrict__ e0dir) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  int64_t k = 0;
  if (in_dirs) {
    d3 u = load3(source) - load3(centers + 3 * p);
    u = div(u, norm(u));
    const int64_t w = wall_ids[p];
    k = brdf_index[w] * S + nearest_direction(in_dirs + w * S * 3, S, u);
  }
  k0[p] = (int32_t)k;
  const int64_t m = spec_dir[k];
  for (int64_t b = 0; b < B; ++b) {
    const double e = energy0[p * B + b];
    for (int64_t d = 0; d < D; ++d)
      e0dir[(p * D + d) * B + b] =
          e * (d == m ? ta[k * B + b] + tc[k * B + b] : ta[k * B + b]);
  }
}

// musum[j,b,t] = sum_d mu[j,d,b,t] for bins t < Tn (float64 sum in direction
// order, float32 result); 8 directions' loads are issued before they are
// added.
__global__ void direction_sum_kernel(int64_t P, int64_t D, int64_t B,
                                     int64_t T, int64_t Tn,
                                     const float *__restrict__ mu,
                                     float *__restrict__ musum) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= P * B * Tn) return;
  const int64_t t = q % Tn, b = (q / Tn) % B, j = q / (B * Tn);
  const float *p = mu + (j * D * B + b) * T + t;  // element (j, 0, b, t)
  const int64_t stride = B * T;                  // next direction
  double s = 0.0;
  int64_t d = 0;
  for (; d + 8 <= D; d += 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = p[(d + k) * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += (double)v[k];
  }
  for (; d < D; ++d) s += (double)p[d * stride];
  musum[(j * B + b) * T + t] = (float)s;
}

// Lane exchanges of a float64 for the reductions below.  swap32 gives a the
// low halves (lanes 0-31) of a and b and b their high halves; swap16 gives a
// the even 16-lane rows and b the odd ones; ror turns each 16-lane row.
__device__ __forceinline__ void swap32(double &a, double &b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a),
                 y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)y,
                                                   false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(
      (uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
  a = __builtin_bit_cast(double, (uint64_t)lo[0] | (uint64_t)hi[0] << 32);
  b = __builtin_bit_cast(double, (uint64_t)lo[1] | (uint64_t)hi[1] << 32);
}
__device__ __forceinline__ void swap16(double &a, double &b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a),
                 y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y,
                                                   false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(
      (uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
  a = __builtin_bit_cast(double, (uint64_t)lo[0] | (uint64_t)hi[0] << 32);
  b = __builtin_bit_cast(double, (uint64_t)lo[1] | (uint64_t)hi[1] << 32);
}
template <int N>
__device__ __forceinline__ double ror(double v) {
  const uint64_t x = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(
      0, (int)(uint32_t)x, 0x120 | N, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(
      0, (int)(uint32_t)(x >> 32), 0x120 | N, 0xf, 0xf, false);
  return __builtin_bit_cast(double, (uint64_t)lo | (uint64_t)hi << 32);
}

// The wave's sums of four values: lanes 0-15 get v0's, 16-31 v2's, 32-47
// v1's, 48-63 v3's (16 vector instructions for each two values; a butterfly
// over the wave for each is 36, 12 of them through LDS).
__device__ __forceinline__ double wave_sums(double v0, double v1, double v2,
                                            double v3) {
  swap32(v0, v1);
  swap32(v2, v3);
  double a = v0 + v1, b = v2 + v3;
  swap16(a, b);
  double s = a + b;
  s += ror<8>(s);
  s += ror<4>(s);
  s += ror<2>(s);
  return s + ror<1>(s);
}

// One backward order: mu_out = lambda + A^T mu_next, and the entries' table
// gradients ga[0,b,q] += sum_t musum[j,b,t+n] ek[i,d',b,t], ga[1,b,q] +=
// sum_t mu_next[j,m,b,t+n] ek[i,d',b,t] (q: transposed entry, d' its source
// direction).  A workgroup of 8 waves takes one (source i, band, block of
// 64 R bins), sources fastest.  It sets its part of mu_out to lambda; then
// each wave sums a run of whole directions with about an eighth of the
// source's entries (sorted by direction, a flag on the last entry of each),
// two at a time, the next two's loads (mu-sum row, specular mu row, the
// source's own order-k row) in flight while the current ones are summed.
// Each lane makes one entry of 64 ready (addresses and bytes left in the
// rows), which the wave then takes by v_readlane.  At a direction's last
// entry the sum is added to its mu_out row with float atomics (each element
// receives exactly one add, so the result does not depend on their order).
// A bin t + n beyond the histogram is an out-of-range buffer offset and reads
// 0.  The dot products of two entries are reduced over the wave at once and
// added (float64 atomics) by four lanes.  Requires T < 2^29.  Only bins that
// E_k can hold energy in (t < Tk) are formed, from mu_next's bins below Tn
// (those of E_{k+1}, at least Tk plus the longest delay or T).
// Bound by the vector instructions of an entry, about 50 of which 28 are its
// sums, and by latency where there are few sources.  232 patches, 64
// directions, 3 bands: 107 us on average over orders of up to 1,400 bins;
// with four waves of 64 R bins that each walked all entries, a butterfly for
// each dot product and lambda copied by a launch of its own 206 + 24 us.
// Gradient of a directional shoebox (1,072 patches, 6 bands, 2,000 bins, 10
// orders) 91 ms instead of 124.
constexpr int kAdjointWaves = 8;

template <int R>
__global__ __launch_bounds__(64 * kAdjointWaves)
    __attribute__((amdgpu_waves_per_eu(4))) void adjoint_ds_kernel(
        int D, int B, int T, int Tk, int Tn, int n_tblk, int64_t nblocks,
        uint32_t first, uint32_t count, int64_t Vd,
        const int64_t *__restrict__ tgptr,
        const int32_t *__restrict__ tkey, const int32_t *__restrict__ tlag,
        const int32_t *__restrict__ tm, const double *__restrict__ twa,
        const double *__restrict__ twc, const float *__restrict__ lam,
        const float *__restrict__ musum, const float *__restrict__ munext,
        const float *__restrict__ ek, float *__restrict__ muout,
        double *__restrict__ ga) {
  constexpr int NW = kAdjointWaves, TB = 64 * R, C = 2;
  constexpr int32_t kDstMask = (1 << 25) - 1;
  int64_t i;
  int b, tb;
  dest_major_tile(first + xcd_tile(blockIdx.x, count), nblocks, B, n_tblk,
                  i, b, tb);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const int t0 = tb * TB;
  const int64_t srow = i * D;  // row (i, d') = srow + d'
  const int64_t stride = (int64_t)B * T;

  // mu_out = lambda: the waves take the directions in turn
  const int64_t own = srow * stride + (int64_t)b * T + t0;
  const uint32_t own_bytes = (uint32_t)min(Tk - t0, TB) * 4u;
  constexpr int CP = 4;  // rows' loads in flight
  for (int d = wave; d < D; d += NW * CP) {
    float v[CP][R];
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int dd = d + c * NW;
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc(lam + own + min(dd, D - 1) * stride,
                    dd < D ? own_bytes : 0u);
#pragma unroll
      for (int r = 0; r < R; ++r)
        v[c][r] = buffer_load(rs, (uint32_t)(lane + 64 * r) * 4u);
    }
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int dd = d + c * NW;
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc(muout + own + min(dd, D - 1) * stride,
                    dd < D ? own_bytes : 0u);
#pragma unroll
      for (int r = 0; r < R; ++r)
        buffer_store(v[c][r], rs, (uint32_t)(lane + 64 * r) * 4u);
    }
  }

  // the wave's entries [e_lo, e_hi): whole directions whose first entry lies
  // in the wave's eighth
  const int64_t *starts = tgptr + srow;
  const int64_t q0 = starts[0], q1 = starts[D];
  const int64_t cut_lo = q0 + (q1 - q0) * wave / NW;
  const int64_t cut_hi = q0 + (q1 - q0) * (wave + 1) / NW;
  int64_t e_lo = q1, e_hi = q1;
  for (int d = 0; d < D; d += 64) {
    const bool in = d + lane < D;
    const int64_t st = starts[in ? d + lane : D];
    const uint64_t lo = __ballot(in && st >= cut_lo);
    const uint64_t hi = __ballot(in && st >= cut_hi);
    if (lo != 0 && e_lo == q1) e_lo = readlane_i64(st, __builtin_ctzll(lo));
    if (hi != 0 && e_hi == q1) e_hi = readlane_i64(st, __builtin_ctzll(hi));
  }
  // the stores above are complete (vmcnt(0): in the L2 that this workgroup's
  // atomics work in) before any wave adds to them
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (e_hi <= e_lo) return;  // uniform, after the barrier

  const double *wa = twa + (int64_t)b * Vd, *wc = twc + (int64_t)b * Vd;
  double *gda = ga + (int64_t)b * Vd, *gdc = ga + ((int64_t)B + b) * Vd;
  struct Meta {
    int32_t key, lag, m;
    double a, c;
  };
  struct Ready {
    int64_t x, y, row;  // addresses; the source's row from ek's first element
    int32_t bytes;
    double a, c;
    uint64_t ends;
  };
  auto load_meta = [&](int64_t e0) {
    const int64_t q = e0 + lane;
    const bool in = q < e_hi;
    const int64_t qc = in ? q : e_hi - 1;
    Meta v;
    v.key = tkey[qc];
    v.m = tm[qc];
    v.lag = in ? tlag[qc] : kLagMask;  // past the end: no bins, no flag
    v.a = in ? wa[qc] : 0.0;
    v.c = in ? wc[qc] : 0.0;
    return v;
  };
  auto ready = [&](const Meta &v) {
    Ready x;
    const int64_t j = v.key & kDstMask, d = v.key >> 25;
    const int n = min(v.lag & kLagMask, T), first = t0 + n;
    x.x = (int64_t)(musum + (j * B + b) * (int64_t)T + first);
    x.y = (int64_t)(munext + ((j * D + v.m) * B + b) * (int64_t)T + first);
    x.row = ((srow + d) * B + b) * (int64_t)T + t0;
    x.bytes = max(Tn - first, 0) * 4;
    x.a = v.a;
    x.c = v.c;
    x.ends = __ballot((v.lag & kLastInGroup) != 0);
    return x;
  };
  auto fetch = [&](const Ready &v, int q, float (&x)[C][R], float (&y)[C][R],
                   float (&e)[C][R]) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint32_t sz =
          (uint32_t)__builtin_amdgcn_readlane(v.bytes, q + c);
      const __amdgpu_buffer_rsrc_t rx =
          make_rsrc((const void *)readlane_i64(v.x, q + c), sz);
      const __amdgpu_buffer_rsrc_t ry =
          make_rsrc((const void *)readlane_i64(v.y, q + c), sz);
      const __amdgpu_buffer_rsrc_t re =
          make_rsrc(ek + readlane_i64(v.row, q + c), own_bytes);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t off = (uint32_t)lane * 4u + 256u * (uint32_t)r;
        x[c][r] = buffer_load(rx, off);
        y[c][r] = buffer_load(ry, off);
        e[c][r] = buffer_load(re, off);
      }
    }
  };
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  auto consume = [&](const Ready &v, int64_t blk, int q,
                     const float (&x)[C][R], const float (&y)[C][R],
                     const float (&e)[C][R]) {
    double pa[C], pc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      pa[c] = pc[c] = 0.0;
      const double wx = readlane_f64(v.a, q + c);
      const double wy = readlane_f64(v.c, q + c);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double xd = (double)x[c][r], yd = (double)y[c][r];
        const double ed = (double)e[c][r];
        acc[r] = fma(wx, xd, acc[r]);
        acc[r] = fma(wy, yd, acc[r]);
        pa[c] = fma(ed, xd, pa[c]);
        pc[c] = fma(ed, yd, pc[c]);
      }
      if ((v.ends >> (q + c) & 1ull) != 0) {  // uniform
        float *o = muout + readlane_i64(v.row, q + c) + lane;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (t0 + lane + 64 * r < Tk)
            unsafeAtomicAdd(o + 64 * r, (float)acc[r]);
          acc[r] = 0.0;
        }
      }
    }
    const double sum = wave_sums(pa[0], pa[1], pc[0], pc[1]);
    const int64_t qq = blk + q + (lane >> 5);
    if ((lane & 15) == 0 && qq < e_hi)
      unsafeAtomicAdd((lane & 16 ? gdc : gda) + qq, sum);
  };
  Meta next = load_meta(e_lo);
  float xa[C][R], ya[C][R], ea[C][R], xb[C][R], yb[C][R], eb[C][R];
  for (int64_t blk = e_lo; blk < e_hi; blk += 64) {
    const Ready cur = ready(next);
    next = load_meta(blk + 64);
    const int n = (int)min((int64_t)64, e_hi - blk);
    fetch(cur, 0, xa, ya, ea);
    for (int q = 0; q < n; q += 2 * C) {
      if (q + C < n) fetch(cur, q + C, xb, yb, eb);
      consume(cur, blk, q, xa, ya, ea);
      if (q + C >= n) break;
      if (q + 2 * C < n) fetch(cur, q + 2 * C, xa, ya, ea);
      consume(cur, blk, q + C, xb, yb, eb);
    }
  }
}

// Table gradients from the entries' accumulated dot products:
// gA[k,b] += wgt[b,e] ga[0,b,q], gC[k,b] += wgt[b,e] ga[1,b,q] with
// e = te[q], k = krow[e].
__global__ void table_grad_kernel(int64_t B, int64_t Vd,
                                  const int32_t *__restrict__ te,
                                  const int32_t *__restrict__ krow,
                                  const double *__restrict__ wgt,
                                  const double *__restrict__ ga,
                                  double *__restrict__ gA,
                                  double *__restrict__ gC) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= B * Vd) return;
  const int64_t b = q / Vd, p = q % Vd;
  const int64_t e = te[p];
  const int64_t k = krow[e];
  const double w = wgt[b * Vd + e];
  unsafeAtomicAdd(gA + k * B + b, w * ga[q]);
  unsafeAtomicAdd(gC + k * B + b, w * ga[B * Vd + q]);
}

// Injection gradient: dL/de0dir[p,d,b] = mu0[p,d,b,n_p] with n_p the
// order-0 bin of patch p; gA[k0_p,b] += energy0[p,b] sum_d mu0[p,d,b,n_p],
// gC[k0_p,b] += energy0[p,b] mu0[p,m,b,n_p].
__global__ void injection_grad_kernel(
    int64_t P, int64_t D, int64_t B, int64_t T,
    const double *__restrict__ energy0, const double *__restrict__ d0,
    double c, double dt, const int32_t *__restrict__ k0,
    const int32_t *__restrict__ spec_dir, const float *__restrict__ mu0,
    double *__restrict__ gA, double *__restrict__ gC) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= P * B) return;
  const int64_t p = q / B, b = q % B;
  const int64_t n = delay_floor(d0[p], c, dt);
  if (n < 0 || n >= T) return;
  const int64_t k = k0[p], m = spec_dir[k];
  double s = 0.0, sm = 0.0;
  for (int64_t d = 0; d < D; ++d) {
    const double v = mu0[((p * D + d) * B + b) * T + n];
    s += v;
    if (d == m) sm = v;
  }
  const double e = energy0[p * B + b];
  unsafeAtomicAdd(gA + k * B + b, e * s);
  if (m < D) unsafeAtomicAdd(gC + k * B + b, e * sm);
}

// ---------------------------------------------------------------------
// Adjoint of the grouped plan (any BRDF rows)
// ---------------------------------------------------------------------
// One forward order on the grouped plan (exchange.hip, RadiosityFast.py:
// 1114-1143 grouped by BRDF row):
//   gsum[g,b,t] = sum_{e in g} scal[b,e] E_k[row_e, b, t - n_e],
//   E_{k+1}[j,d,b,t] = sum_{g of j} rtab[key_g, b, d] gsum[g,b,t],
// with rtab[k,b,d] = table[k,d,b] (BRDF row k = brdf * S + s).  For
// mu = dL/dE_{k+1}:
//   nu[g,b,t] = sum_d rtab[key_g,b,d] mu[j_g,d,b,t]              (spread^T)
//   dL/dE_k[r,b,t] += sum_{e: row_e = r} scal[b,e] nu[g_e,b,t+n_e] (gather^T)
//   dL/dtable[key_g,d,b] += sum_t mu[j_g,d,b,t] gsum[g,b,t].

// nu for every group of destination j with up to 8 (padded) directions: a
// workgroup per (j, band, 256 bins), one bin per lane; the lane keeps
// mu[j,:,b,t] as DPT doubles (converted once), and the workgroup stages its
// groups' BRDF rows in LDS, 16 at a time, read by broadcast.  (With 16 or
// more directions grouped_spread_adjoint_mfma_kernel forms nu; this kernel
// took 12.2 ms per call on the directional shoebox.)
template <int DPT>
__global__ __launch_bounds__(256) void grouped_spread_adjoint_kernel(
    int D, int B, int T, int Tn, int DP, int n_tblk,
    const int64_t *__restrict__ grp_ptr, const int32_t *__restrict__ grp_key,
    const double *__restrict__ rtab, const float *__restrict__ mu,
    float *__restrict__ nu) {
  constexpr int NG = 16;
  __shared__ double rts[NG][DPT];
  const int64_t blk = blockIdx.x;
  const int tb = (int)(blk % n_tblk);
  const int b = (int)((blk / n_tblk) % B);
  const int64_t j = blk / ((int64_t)n_tblk * B);
  const int64_t g0 = grp_ptr[j], g1 = grp_ptr[j + 1];
  if (g0 == g1) return;  // uniform
  const int t = tb * 256 + (int)threadIdx.x;
  const bool in = t < Tn;
  const int64_t dstride = (int64_t)B * T;
  const float *m = mu + (j * D * B + b) * (int64_t)T + (in ? t : 0);
  double v[DPT];
#pragma unroll
  for (int d = 0; d < DPT; ++d)
    v[d] = (d < D && in) ? (double)m[d * dstride] : 0.0;
  for (int64_t gc = g0; gc < g1; gc += NG) {
    const int ng = (int)min((int64_t)NG, g1 - gc);
    for (int idx = (int)threadIdx.x; idx < NG * DPT; idx += 256) {
      const int gi = idx / DPT, d = idx % DPT;
      rts[gi][d] = (gi < ng && d < DP)
                       ? rtab[((int64_t)grp_key[gc + gi] * B + b) * DP + d]
                       : 0.0;
    }
    __syncthreads();
    for (int gi = 0; gi < ng; ++gi) {
      double s = 0.0;
#pragma unroll
      for (int d = 0; d < DPT; ++d) s = fma(rts[gi][d], v[d], s);
      if (in) nu[((gc + gi) * B + b) * (int64_t)T + t] = (float)s;
    }
    __syncthreads();
  }
}

// gg[g,b,d] += sum_t mu[j_g,d,b,t] gsum[g,b,t] for the groups g of
// destination j: per (j, band) the product of the group sums [G_j x T]
// with mu[j,:,b,:]^T [T x D], on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64: lane l holds A[l & 15][l >> 4], B[l >> 4][l & 15]
// and D[(l >> 4) + 4r][l & 15]).  Tiles of 16 NQ groups x 16 NR directions
// (NQ from the groups left, NR from D); the bins in chunks of 32 staged in
// LDS as float32, both operands read from there; wave q takes group tile
// q against every direction tile (NR accumulators of 16 x 16).  Each
// (group, direction) is summed by one lane in float64 and owned by it: no
// atomics, and the result does not depend on the launch's timing.  The
// directional shoebox's launch takes 5.5 ms (12.0 ms on the vector unit,
// each lane summing NQ x NR pairs; 10.7 ms here without the prefetch of
// the next chunk; 17.8 ms with chunks of 64 bins).
constexpr int kTgChunk = 32;
typedef double mfma_d4 __attribute__((ext_vector_type(4)));

template <int NQ, int NR>
__device__ __forceinline__ void table_grad_tile(
    int D, int B, int T, int Tn, int DP, int b, int64_t gt, int64_t g1,
    const float *__restrict__ mrow, const float *__restrict__ gsum,
    double *__restrict__ gg, float (&sg)[64][kTgChunk + 1],
    float (&sm)[64][kTgChunk + 1]) {
  constexpr int TC = kTgChunk;
  const int tid = (int)threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int kk = lane >> 4, cc = lane & 15;
  const int64_t dstride = (int64_t)B * T;
  mfma_d4 acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = mfma_d4{0.0, 0.0, 0.0, 0.0};
  // 256 lanes stage 8 rows of 32 bins per step; the next chunk's values
  // are loaded into registers while the current chunk is multiplied
  const int col = tid % TC;
  float pg[2 * NQ], pm[2 * NR];
  auto fetch = [&](int t0) {
    const int t = t0 + col;
#pragma unroll
    for (int s = 0; s < 2 * NQ; ++s) {
      const int64_t g = gt + tid / TC + 8 * s;
      pg[s] = (g < g1 && t < Tn) ? gsum[(g * B + b) * (int64_t)T + t] : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 2 * NR; ++s) {
      const int d = tid / TC + 8 * s;
      pm[s] = (d < D && t < Tn) ? mrow[d * dstride + t] : 0.f;
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < Tn; t0 += TC) {
#pragma unroll
    for (int s = 0; s < 2 * NQ; ++s) sg[tid / TC + 8 * s][col] = pg[s];
#pragma unroll
    for (int s = 0; s < 2 * NR; ++s) sm[tid / TC + 8 * s][col] = pm[s];
    __syncthreads();
    if (t0 + TC < Tn) fetch(t0 + TC);  // uniform
    if (wave < NQ) {  // uniform per wave
#pragma unroll 4
      for (int c = 0; c < TC; c += 4) {
        const double a = (double)sg[16 * wave + cc][c + kk];
#pragma unroll
        for (int r = 0; r < NR; ++r)
          acc[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              a, (double)sm[16 * r + cc][c + kk], acc[r], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (wave >= NQ) return;
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t g = gt + 16 * wave + kk + 4 * i;
      const int d = 16 * r + cc;
      if (g < g1 && d < D) gg[(g * B + b) * DP + d] += acc[r][i];
    }
}

template <int NR>
__global__ __launch_bounds__(256) void grouped_table_grad_kernel(
    int D, int B, int T, int Tn, int DP, const int64_t *__restrict__ grp_ptr,
    const float *__restrict__ mu, const float *__restrict__ gsum,
    double *__restrict__ gg) {
  __shared__ float sg[64][kTgChunk + 1];
  __shared__ float sm[64][kTgChunk + 1];
  const int b = (int)(blockIdx.x % B);
  const int64_t j = blockIdx.x / B;
  const int64_t g0 = grp_ptr[j], g1 = grp_ptr[j + 1];
  const float *mrow = mu + (j * D * B + b) * (int64_t)T;  // (j, 0, b, 0)
  for (int64_t gt = g0; gt < g1; gt += 64) {
    const int64_t left = g1 - gt;  // uniform
    if (left > 48)
      table_grad_tile<4, NR>(D, B, T, Tn, DP, b, gt, g1, mrow, gsum, gg, sg,
                             sm);
    else if (left > 32)
      table_grad_tile<3, NR>(D, B, T, Tn, DP, b, gt, g1, mrow, gsum, gg, sg,
                             sm);
    else if (left > 16)
      table_grad_tile<2, NR>(D, B, T, Tn, DP, b, gt, g1, mrow, gsum, gg, sg,
                             sm);
    else
      table_grad_tile<1, NR>(D, B, T, Tn, DP, b, gt, g1, mrow, gsum, gg, sg,
                             sm);
  }
}

// nu on the FP64 matrix cores (16, 32 or 64 padded directions): per
// destination j and band b the product of the groups' BRDF rows
// [G_j x DP] with mu[j,:,b,:] [DP x T], K = DP in steps of 4.  A workgroup
// per (j, band, 4 x 16 NT bins), each wave 16 NT bins (NT = 2 at 64
// directions, so that the operands fit four waves per SIMD, else 4): the
// wave's mu operands (lane
// l: direction 4s + (l >> 4), bin l & 15 of each 16-bin tile) are loaded
// once into registers, then every tile of 16 groups is multiplied against
// them, its BRDF rows staged in LDS.  Lane layout of
// v_mfma_f64_16x16x4f64 as in grouped_table_grad_kernel.
template <int DP>
struct SpreadAdjMfma {
  static constexpr int NT = DP == 64 ? 2 : 4;  // 16-bin tiles per wave
  static constexpr int BINS = 4 * 16 * NT;      // bins per workgroup
};

template <int DP>
__global__ __launch_bounds__(256) void grouped_spread_adjoint_mfma_kernel(
    int D, int B, int T, int Tn, int n_tblk, const int64_t *__restrict__ grp_ptr,
    const int32_t *__restrict__ grp_key, const double *__restrict__ rtab,
    const float *__restrict__ mu, float *__restrict__ nu) {
  constexpr int KS = DP / 4, NT = SpreadAdjMfma<DP>::NT;
  __shared__ double rts[16][DP + 1];
  const int64_t blk = blockIdx.x;
  const int tb = (int)(blk % n_tblk);
  const int b = (int)((blk / n_tblk) % B);
  const int64_t j = blk / ((int64_t)n_tblk * B);
  const int64_t g0 = grp_ptr[j], g1 = grp_ptr[j + 1];
  if (g0 == g1) return;  // uniform
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, kk = lane >> 4, cc = lane & 15;
  const int tw = (tb * 4 + (tid >> 6)) * 16 * NT;
  const int64_t dstride = (int64_t)B * T;
  const float *m = mu + (j * D * B + b) * (int64_t)T;  // (j, 0, b, 0)
  float mv[KS][NT];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int d = 4 * s + kk, t = tw + 16 * nt + cc;
      const bool ok = d < D && t < Tn;
      const float v = m[ok ? d * dstride + t : 0];
      mv[s][nt] = ok ? v : 0.f;
    }
  for (int64_t gt = g0; gt < g1; gt += 16) {
    for (int idx = tid; idx < 16 * DP; idx += 256) {
      const int gi = idx / DP, d = idx % DP;
      rts[gi][d] = (gt + gi < g1 && d < D)
                       ? rtab[((int64_t)grp_key[gt + gi] * B + b) * DP + d]
                       : 0.0;
    }
    __syncthreads();
    mfma_d4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const double a = rts[cc][4 * s + kk];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(
            a, (double)mv[s][nt], acc[nt], 0, 0, 0);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t g = gt + kk + 4 * r;
        const int t = tw + 16 * nt + cc;
        if (g < g1 && t < Tn)
          nu[(g * B + b) * (int64_t)T + t] = (float)acc[nt][r];
      }
    __syncthreads();
  }
}

// muout[r,b,t] = lam[r,b,t] + sum_{q in T(r)} tscal[b,q] nu[tgrp_q,b,t+n_q]
// for bins t < Tk (float64 sum in transposed-entry order; a bin t + n from Tn
// on reads 0 through the row's buffer descriptor and adds nothing).  A
// workgroup per (source row r, band, 256 R bins), R bins per lane, rows
// taken direction-major (r = i*D + d for d slow, i fast: neighbouring
// patches sending in one direction feed the same groups, whose nu rows
// they then share through L2); the entries are taken C at a time, every
// load of the chunk issued before any is summed.
template <int R>
__global__ __launch_bounds__(256) void grouped_gather_adjoint_kernel(
    int64_t P, int D, int B, int T, int Tk, int Tn, int n_tblk, int64_t Vd,
    const int64_t *__restrict__ trow_ptr,
    const int32_t *__restrict__ tgrp, const int32_t *__restrict__ tlag,
    const double *__restrict__ tscal, const float *__restrict__ nu,
    const float *__restrict__ lam, float *__restrict__ muout) {
  constexpr int C = 4;
  const int64_t blk = blockIdx.x;
  const int tb = (int)(blk % n_tblk);
  const int b = (int)((blk / n_tblk) % B);
  const int64_t rd = blk / ((int64_t)n_tblk * B);  // d * P + i
  const int64_t r = (rd % P) * D + rd / P;
  const int64_t q0 = trow_ptr[r], q1 = trow_ptr[r + 1];
  const int64_t base = (r * B + b) * (int64_t)T;
  const uint32_t row_bytes = (uint32_t)Tn * 4u;
  int t[R];
  double s[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    t[i] = tb * 256 * R + (int)threadIdx.x + 256 * i;
    s[i] = t[i] < Tk ? (double)lam[base + t[i]] : 0.0;
  }
  for (int64_t q = q0; q < q1; q += C) {
    float v[C][R];
    double w[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = q + c < q1;  // uniform
      const int64_t qq = ok ? q + c : q0;
      const int n = tlag[qq];
      w[c] = ok ? tscal[b * Vd + qq] : 0.0;
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(
          nu + ((int64_t)tgrp[qq] * B + b) * (int64_t)T, ok ? row_bytes : 0u);
#pragma unroll
      for (int i = 0; i < R; ++i) v[c][i] = buffer_load(rs, bin_offset(t[i] + n));
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (q + c >= q1) break;  // uniform
#pragma unroll
      for (int i = 0; i < R; ++i) s[i] = fma(w[c], (double)v[c][i], s[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (t[i] < Tk) muout[base + t[i]] = (float)s[i];
}

// gt[key_g,d,b] += gg[g,b,d] (float64 atomics: the groups of one BRDF row
// add in no fixed order).
__global__ void grouped_key_grad_kernel(int64_t G, int D, int B, int DP,
                                        const int32_t *__restrict__ grp_key,
                                        const double *__restrict__ gg,
                                        double *__restrict__ gt) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= G * B * D) return;
  const int d = (int)(q % D);
  const int b = (int)((q / D) % B);
  const int64_t g = q / ((int64_t)D * B);
  unsafeAtomicAdd(gt + ((int64_t)grp_key[g] * D + d) * B + b,
                  gg[(g * B + b) * DP + d]);
}

// Injection part: E_0dir[p,d,b] = energy0[p,b] table[k0_p,d,b], placed at
// bin n_p, so gt[k0_p,d,b] += energy0[p,b] mu0[p,d,b,n_p].
__global__ void injection_table_grad_kernel(
    int64_t P, int64_t D, int64_t B, int64_t T,
    const double *__restrict__ energy0, const double *__restrict__ d0,
    double c, double dt, const int32_t *__restrict__ k0,
    const float *__restrict__ mu0, double *__restrict__ gt) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= P * D * B) return;
  const int64_t b = q % B, d = (q / B) % D, p = q / (D * B);
  const int64_t n = delay_floor(d0[p], c, dt);
  if (n < 0 || n >= T) return;
  unsafeAtomicAdd(gt + ((int64_t)k0[p] * D + d) * B + b,
                  energy0[p * B + b] * (double)mu0[q * T + n]);
}

}  // namespace

int direction_sum(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
                  const float *mu, float *musum, hipStream_t s) {
  hipLaunchKernelGGL(direction_sum_kernel,
                     dim3((unsigned)ceil_div(P * B * Tn, 256)), dim3(256), 0,
                     s, P, D, B, T, Tn, mu, musum);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

int adjoint_ds(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tk,
               int64_t Tn, int64_t Vd, const int64_t *tgptr,
               const int32_t *tkey, const int32_t *tlag, const int32_t *tm,
               const double *twa, const double *twc, const float *lam,
               const float *musum, const float *munext, const float *ek,
               float *muout, double *ga, hipStream_t s) {
  auto go = [&](auto kernel, int R) {
    const int64_t nt = ceil_div(Tk, (int64_t)64 * R);
    const int64_t nb = P * B * nt;
    SPR_REQUIRE(nb < (int64_t)0x7fffffff,
                "spr_exchange_adjoint_ds: grid too large");
    // 8 waves for 128 or 256 bins: 8.4 M blocks reach a launch's limit
    const int64_t most = max_blocks(64 * kAdjointWaves);
    for (int64_t first = 0; first < nb; first += most) {
      const uint32_t count = (uint32_t)std::min(most, nb - first);
      hipLaunchKernelGGL(kernel, dim3(count), dim3(64 * kAdjointWaves), 0, s,
                         (int)D, (int)B, (int)T, (int)Tk, (int)Tn, (int)nt, nb,
                         (uint32_t)first, count, Vd, tgptr, tkey, tlag, tm,
                         twa, twc, lam, musum, munext, ek, muout, ga);
    }
    SPR_LAUNCH_CHECK();
    return SPR_OK;
  };
  // 4 bins per lane, or 2 where 4 would reach past Tk for nothing: an entry's
  // reductions and lane reads then serve 256 bins (8 do not fit the
  // registers).
  if (Tk <= 128) return go(adjoint_ds_kernel<2>, 2);
  return go(adjoint_ds_kernel<4>, 4);
}

int spread_adjoint(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
                   const int64_t *grp_ptr, const int32_t *grp_key,
                   const double *rtab, const float *mu, float *nu,
                   hipStream_t s) {
  const int64_t DP = spr_padded_directions(D);
  const int64_t nt = ceil_div(Tn, (int64_t)256);
  const int64_t nb = P * B * nt;
  SPR_REQUIRE(2 * nb < (int64_t)0x7fffffff,  // 128-bin blocks at D = 64
              "spr_grouped_spread_adjoint: grid too large");
  auto mfma = [&](auto kernel, int64_t bins) {
    const int64_t n = ceil_div(Tn, bins);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(P * B * n)), dim3(256), 0, s,
                       (int)D, (int)B, (int)T, (int)Tn, (int)n, grp_ptr,
                       grp_key, rtab, mu, nu);
  };
  if (DP == 16)
    mfma(grouped_spread_adjoint_mfma_kernel<16>, SpreadAdjMfma<16>::BINS);
  else if (DP == 32)
    mfma(grouped_spread_adjoint_mfma_kernel<32>, SpreadAdjMfma<32>::BINS);
  else if (DP == 64)
    mfma(grouped_spread_adjoint_mfma_kernel<64>, SpreadAdjMfma<64>::BINS);
  else  // up to 8 directions: the vector kernel
    hipLaunchKernelGGL((grouped_spread_adjoint_kernel<8>), dim3((unsigned)nb),
                       dim3(256), 0, s, (int)D, (int)B, (int)T, (int)Tn,
                       (int)DP, (int)nt, grp_ptr, grp_key, rtab, mu, nu);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

int table_grad(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
               const int64_t *grp_ptr, const float *mu, const float *gsum,
               double *gg, hipStream_t s) {
  const int64_t DP = spr_padded_directions(D);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(P * B)), dim3(256), 0, s,
                       (int)D, (int)B, (int)T, (int)Tn, (int)DP, grp_ptr, mu,
                       gsum, gg);
  };
  if (D <= 16)
    go(grouped_table_grad_kernel<1>);
  else if (D <= 32)
    go(grouped_table_grad_kernel<2>);
  else if (D <= 48)
    go(grouped_table_grad_kernel<3>);
  else
    go(grouped_table_grad_kernel<4>);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

int gather_adjoint(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tk,
                   int64_t Tn, int64_t Vd, const int64_t *trow_ptr,
                   const int32_t *tgrp, const int32_t *tlag,
                   const double *tscal, const float *nu, const float *lam,
                   float *muout, hipStream_t s) {
  auto go = [&](auto kernel, int R) {
    const int64_t nt = ceil_div(Tk, (int64_t)256 * R);
    const int64_t nb = P * D * B * nt;
    SPR_REQUIRE(nb < (int64_t)0x7fffffff,
                "spr_grouped_gather_adjoint: grid too large");
    hipLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(256), 0, s, P, (int)D,
                       (int)B, (int)T, (int)Tk, (int)Tn, (int)nt, Vd, trow_ptr,
                       tgrp, tlag, tscal, nu, lam, muout);
    SPR_LAUNCH_CHECK();
    return SPR_OK;
  };
  if (Tk <= 256) return go(grouped_gather_adjoint_kernel<1>, 1);
  if (Tk <= 512) return go(grouped_gather_adjoint_kernel<2>, 2);
  return go(grouped_gather_adjoint_kernel<4>, 4);
}

}  // namespace spr

using namespace spr;

extern "C" int spr_ds_weights(int64_t B, int64_t Vd, const int32_t *krow,
                              const double *wgt, const double *a,
                              const double *cs, double *scal, double *dscal,
                              void *stream) {
  SPR_REQUIRE(B > 0 && Vd >= 0, "spr_ds_weights: bad sizes");
  SPR_REQUIRE(krow && wgt && a && cs && scal && dscal,
              "spr_ds_weights: null pointer");
  if (Vd == 0) return SPR_OK;
  hipLaunchKernelGGL(ds_weights_kernel, dim3((unsigned)ceil_div(B * Vd, 256)),
                     dim3(256), 0, as_stream(stream), B, Vd, krow, wgt, a, cs,
                     scal, dscal);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_ds_transposed_weights(int64_t B, int64_t Vd,
                                         const int32_t *te,
                                         const double *scal,
                                         const double *dscal, double *twa,
                                         double *twc, void *stream) {
  SPR_REQUIRE(B > 0 && Vd >= 0, "spr_ds_transposed_weights: bad sizes");
  SPR_REQUIRE(te && scal && dscal && twa && twc,
              "spr_ds_transposed_weights: null pointer");
  if (Vd == 0) return SPR_OK;
  hipLaunchKernelGGL(t_weights_kernel, dim3((unsigned)ceil_div(B * Vd, 256)),
                     dim3(256), 0, as_stream(stream), B, Vd, te, scal, dscal,
                     twa, twc);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_ds_injection(int64_t P, int64_t D, int64_t B,
                                const double *source, const double *centers,
                                const int64_t *wall_ids, int64_t S,
                                const int64_t *brdf_index,
                                const double *in_dirs, const double *energy0,
                                const double *a, const double *cs,
                                const int32_t *spec_dir, int32_t *k0,
                                double *e0dir, void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && B > 0, "spr_ds_injection: bad sizes");
  SPR_REQUIRE(source && centers && energy0 && a && cs && spec_dir && k0 &&
                  e0dir,
              "spr_ds_injection: null pointer");
  SPR_REQUIRE(!in_dirs || (wall_ids && brdf_index && S > 0),
              "spr_ds_injection: in_dirs needs wall_ids, brdf_index");
  hipLaunchKernelGGL(ds_injection_kernel, dim3((unsigned)ceil_div(P, 128)),
                     dim3(128), 0, as_stream(stream), P, D, B, source, centers,
                     wall_ids, S, brdf_index, in_dirs, energy0, a, cs,
                     spec_dir, k0, e0dir);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_direction_sum(int64_t P, int64_t D, int64_t B, int64_t T,
                                 const float *mu, float *musum,
                                 void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && B > 0 && T > 0,
              "spr_direction_sum: bad sizes");
  SPR_REQUIRE(mu && musum, "spr_direction_sum: null pointer");
  return direction_sum(P, D, B, T, T, mu, musum, as_stream(stream));
}

extern "C" int spr_exchange_adjoint_ds(
    int64_t P, int64_t D, int64_t B, int64_t T, int64_t Vd,
    const int64_t *tgptr, const int32_t *tkey, const int32_t *tlag,
    const int32_t *tm, const double *twa, const double *twc,
    const float *lam, const float *musum, const float *munext,
    const float *ek, float *muout, double *ga, void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && D <= 64 && B > 0 && T > 0 && Vd >= 0,
              "spr_exchange_adjoint_ds: bad sizes");
  SPR_REQUIRE(T < ((int64_t)1 << 29) && P < ((int64_t)1 << 25),
              "spr_exchange_adjoint_ds: histogram or scene too large");
  SPR_REQUIRE(tgptr && tkey && tlag && tm && twa && twc && lam && musum &&
                  munext && ek && muout && ga,
              "spr_exchange_adjoint_ds: null pointer");
  SPR_REQUIRE(muout != munext && muout != lam && muout != ek,
              "spr_exchange_adjoint_ds: muout aliases an input");
  return adjoint_ds(P, D, B, T, T, T, Vd, tgptr, tkey, tlag, tm, twa, twc, lam,
                    musum, munext, ek, muout, ga, as_stream(stream));
}

extern "C" int spr_ds_table_grad(int64_t B, int64_t Vd, const int32_t *te,
                                 const int32_t *krow, const double *wgt,
                                 const double *ga, double *gA, double *gC,
                                 void *stream) {
  SPR_REQUIRE(B > 0 && Vd >= 0, "spr_ds_table_grad: bad sizes");
  SPR_REQUIRE(te && krow && wgt && ga && gA && gC,
              "spr_ds_table_grad: null pointer");
  if (Vd == 0) return SPR_OK;
  hipLaunchKernelGGL(table_grad_kernel, dim3((unsigned)ceil_div(B * Vd, 256)),
                     dim3(256), 0, as_stream(stream), B, Vd, te, krow, wgt, ga,
                     gA, gC);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_ds_injection_grad(int64_t P, int64_t D, int64_t B,
                                     int64_t T, const double *energy0,
                                     const double *d0, double c, double dt,
                                     const int32_t *k0,
                                     const int32_t *spec_dir,
                                     const float *mu0, double *gA,
                                     double *gC, void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && B > 0 && T > 0 && c > 0 && dt > 0,
              "spr_ds_injection_grad: bad sizes");
  SPR_REQUIRE(energy0 && d0 && k0 && spec_dir && mu0 && gA && gC,
              "spr_ds_injection_grad: null pointer");
  hipLaunchKernelGGL(injection_grad_kernel,
                     dim3((unsigned)ceil_div(P * B, 256)), dim3(256), 0,
                     as_stream(stream), P, D, B, T, energy0, d0, c, dt, k0,
                     spec_dir, mu0, gA, gC);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_grouped_spread_adjoint(int64_t P, int64_t D, int64_t B,
                                          int64_t T, const int64_t *grp_ptr,
                                          const int32_t *grp_key,
                                          const double *rtab, const float *mu,
                                          float *nu, void *stream) {
  const int64_t DP = spr_padded_directions(D);
  SPR_REQUIRE(P > 0 && DP > 0 && B > 0 && T > 0 && T < ((int64_t)1 << 29),
              "spr_grouped_spread_adjoint: bad sizes");
  SPR_REQUIRE(grp_ptr && grp_key && rtab && mu && nu,
              "spr_grouped_spread_adjoint: null pointer");
  return spread_adjoint(P, D, B, T, T, grp_ptr, grp_key, rtab, mu, nu,
                        as_stream(stream));
}

extern "C" int spr_grouped_table_grad(int64_t P, int64_t D, int64_t B,
                                      int64_t T, const int64_t *grp_ptr,
                                      const float *mu, const float *gsum,
                                      double *gg, void *stream) {
  const int64_t DP = spr_padded_directions(D);
  SPR_REQUIRE(P > 0 && DP > 0 && B > 0 && T > 0 && T < ((int64_t)1 << 29),
              "spr_grouped_table_grad: bad sizes");
  SPR_REQUIRE(grp_ptr && mu && gsum && gg,
              "spr_grouped_table_grad: null pointer");
  SPR_REQUIRE(P * B < (int64_t)0x7fffffff,
              "spr_grouped_table_grad: grid too large");
  return table_grad(P, D, B, T, T, grp_ptr, mu, gsum, gg, as_stream(stream));
}

extern "C" int spr_grouped_gather_adjoint(
    int64_t P, int64_t D, int64_t B, int64_t T, int64_t Vd,
    const int64_t *trow_ptr, const int32_t *tgrp, const int32_t *tlag,
    const double *tscal, const float *nu, const float *lam, float *muout,
    void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && B > 0 && T > 0 && Vd >= 0 &&
                  T < ((int64_t)1 << 29),
              "spr_grouped_gather_adjoint: bad sizes");
  SPR_REQUIRE(trow_ptr && tgrp && tlag && tscal && nu && lam && muout,
              "spr_grouped_gather_adjoint: null pointer");
  SPR_REQUIRE(muout != lam, "spr_grouped_gather_adjoint: muout aliases lam");
  return gather_adjoint(P, D, B, T, T, T, Vd, trow_ptr, tgrp, tlag, tscal, nu,
                        lam, muout, as_stream(stream));
}

extern "C" int spr_grouped_key_grad(int64_t G, int64_t D, int64_t B,
                                    const int32_t *grp_key, const double *gg,
                                    double *gt, void *stream) {
  const int64_t DP = spr_padded_directions(D);
  SPR_REQUIRE(G >= 0 && DP > 0 && B > 0, "spr_grouped_key_grad: bad sizes");
  SPR_REQUIRE(grp_key && gg && gt, "spr_grouped_key_grad: null pointer");
  if (G == 0) return SPR_OK;
  hipLaunchKernelGGL(grouped_key_grad_kernel,
                     dim3((unsigned)ceil_div(G * B * D, 256)), dim3(256), 0,
                     as_stream(stream), G, (int)D, (int)B, (int)DP, grp_key,
                     gg, gt);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

extern "C" int spr_injection_table_grad(int64_t P, int64_t D, int64_t B,
                                        int64_t T, const double *energy0,
                                        const double *d0, double c, double dt,
                                        const int32_t *k0, const float *mu0,
                                        double *gt, void *stream) {
  SPR_REQUIRE(P > 0 && D > 0 && B > 0 && T > 0 && c > 0 && dt > 0,
              "spr_injection_table_grad: bad sizes");
  SPR_REQUIRE(energy0 && d0 && k0 && mu0 && gt,
              "spr_injection_table_grad: null pointer");
  hipLaunchKernelGGL(injection_table_grad_kernel,
                     dim3((unsigned)ceil_div(P * D * B, 256)), dim3(256), 0,
                     as_stream(stream), P, D, B, T, energy0, d0, c, dt, k0,
                     mu0, gt);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}
