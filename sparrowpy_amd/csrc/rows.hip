// One reflection order in one launch: group sums and their spread over the
// directions, a destination's group sums staying in LDS.
//
// Reference: the per-order loop of _energy_exchange
// (sparrowpy/classes/RadiosityFast.py:1073-1145), as grouped by
// spr_plan_grouped_sort / _fill and spr_plan_ds_sort / _fill.
//
// The two-pass order (gather on destination tiles, then spread) is made for
// large scenes: a tile's workgroup walks the sources of 16 destinations in
// turn, so a room of ten tiles keeps twenty workgroups busy for as long as
// one of them takes.  Here a workgroup of 8 waves takes one destination,
// band and block of 64 R bins, and its waves share the destination's groups:
// a 228-patch room (16 directions, 1 band, 700 bins) takes 35 us per order
// instead of 127, launches included, a 508-patch one (3 bands, 1,500 bins)
// 350 instead of 449.  Large scenes stay with the tiles, which read a source
// row once for 16 destinations (1,072 patches, 8 bands, 1,500 bins: 2.6 ms
// against 3.0).
#include <algorithm>
#include <cmath>

#include "spr_common.hpp"
#include "spr_exchange.hpp"

namespace spr {
namespace {

constexpr int kRowWaves = 8;

struct RowArgs {
  int D, B, T, n_tblk;
  int64_t nblocks, Vd;
  OrderSpan sp;
  Injection inj;  // order of the running sum (n0 set), else none
  int max_groups;
  const int64_t *row_ptr, *grp_ptr, *grp_start;
  const int32_t *grp_key, *rowid, *lag;
  const double *scal, *dscal, *rtab;
  const float *prev;      // source histograms
  const float *pair;      // added to the total with this order, or null
  float *cur, *tot_hi, *tot_lo;  // no total: null; group sums only: all null
  float *gsum;                   // the group sums for the adjoint, or null
};

// LDS bytes of a workgroup: the group sums, and, where the waves share a sum
// (the diffuse sum, or a destination's only group), its parts; then the
// groups' BRDF rows, or the direction map of the diffuse + specular plan.
inline size_t row_lds(const spr_exchange_plan &p, int R) {
  const bool ds = p.kind == SPR_PLAN_DS;
  size_t n = (size_t)p.max_groups * 64 * R * sizeof(float);
  if (ds || p.max_groups == 1) n += (size_t)kRowWaves * 64 * R * sizeof(double);
  return n + (ds ? 64 * sizeof(int32_t)
                 : (size_t)p.max_groups * spr_padded_directions(p.D) *
                       sizeof(double));
}

// Phase 1: each wave sums a run of whole groups with about an eighth of the
// entries, C entries' rows in flight at a time (metadata one entry per lane,
// broadcast with v_readlane), in float64, and writes each group's sum to
// LDS as float32 -- the sums the two-pass order stores, bit for bit, save
// those that the waves share (the diffuse sum, a plan's only group): 8 parts
// in float64, whose sum may round to the other neighbour.  Phase 2:
// each wave sums the groups times their BRDF rows for its directions, in
// group order, in float64, and writes the order and the total.
// Bound by the row reads: an entry's R = 4 loads take 16 clocks of the CU's
// first-level cache, its 13 vector instructions as many.  Forming each
// entry's row address and offsets in the wave (23 scalar and 6 vector
// instructions more) a 328-patch, 4-band order took 139 us instead of 126.
// With two weights and 64 directions the second phase is half of it; its
// values are picked where they are written, 16 totals' loads in flight
// (1,072 patches, 6 bands: 7.0 ms, with the values held in registers and 8
// loads in flight 7.3).  Four waves per SIMD (two workgroups per CU) at up to
// 128 registers.
template <int DP, int R, bool DS>
__global__ __launch_bounds__(64 * kRowWaves)
    __attribute__((amdgpu_waves_per_eu(4))) void row_order_kernel(RowArgs a) {
  constexpr int NW = kRowWaves, TB = 64 * R, C = 16 / R;
  extern __shared__ char smem[];
  float *gs = reinterpret_cast<float *>(smem);  // [max_groups][TB]
  double *part = reinterpret_cast<double *>(gs + (size_t)a.max_groups * TB);
  const int B = a.B, D = a.D;
  const int64_t T = a.T;
  int64_t j;
  int b, tb;
  dest_major_tile(xcd_tile(blockIdx.x, a.nblocks), a.nblocks, B, a.n_tblk, j,
                  b, tb);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const int t0 = tb * TB, t_end = min(a.sp.Tc, t0 + TB);
  const int tl = t0 + lane;
  const int64_t e_begin = a.row_ptr[j], e_end = a.row_ptr[j + 1];
  const int64_t g0 = a.grp_ptr[j];
  const int ng = (int)(a.grp_ptr[j + 1] - g0);
  const bool one = !DS && a.max_groups == 1;  // the waves share the group
  double *ct = part + (one ? NW * TB : 0);    // [max_groups][DP], !DS
  const double *w = a.scal + (int64_t)b * a.Vd;
  const double *w2 = DS ? a.dscal + (int64_t)b * a.Vd : w;

  // the wave's groups [c_lo, c_hi) and entries [e_lo, e_hi): whole groups
  // whose start lies in the wave's eighth of the entries
  const int64_t cut_lo = e_begin + (e_end - e_begin) * wave / NW;
  const int64_t cut_hi = e_begin + (e_end - e_begin) * (wave + 1) / NW;
  auto start_of = [&](int g) -> int64_t {
    return a.grp_start ? a.grp_start[g0 + g] : a.grp_key[g0 + g];
  };
  int c_lo = 0, c_hi = 0;
  for (int i = 0; i < ng; i += 64) {
    const bool in = i + lane < ng;
    const int64_t st = start_of(in ? i + lane : ng - 1);
    c_lo += __popcll(__ballot(in && st < cut_lo));
    c_hi += __popcll(__ballot(in && st < cut_hi));
  }
  if (wave == NW - 1) c_hi = ng;
  // (the diffuse group starts at the row's end: where a destination's entries
  // all lack a specular direction it is the only one, and shared as well)
  const bool share = one || (DS && ng == 1);
  const int64_t e_lo = share       ? cut_lo
                       : c_lo < ng ? start_of(c_lo)
                                   : e_end;
  const int64_t e_hi = share                        ? cut_hi
                       : c_hi < ng && wave < NW - 1 ? start_of(c_hi)
                                                    : e_end;

  if (!DS) {
    for (int i = (int)threadIdx.x; i < ng * DP; i += 64 * NW)
      ct[i] = a.rtab[((int64_t)a.grp_key[g0 + i / DP] * B + b) * DP + i % DP];
  } else {
    int32_t *gmap = reinterpret_cast<int32_t *>(part + (size_t)NW * TB);
    for (int d = (int)threadIdx.x; d < DP; d += 64 * NW) gmap[d] = -1;
    __syncthreads();
    for (int g = (int)threadIdx.x; g < ng - 1; g += 64 * NW) {
      const int32_t k = a.grp_key[g0 + g];
      if (k >= 0 && k < D) gmap[k] = g;
    }
  }

  double S[R], Sd[DS ? R : 1];
#pragma unroll
  for (int r = 0; r < R; ++r) S[r] = 0.0;
#pragma unroll
  for (int r = 0; r < (DS ? R : 1); ++r) Sd[r] = 0.0;
  int gl = c_lo;
  // One entry per lane, 64 at a time: as loaded (a block ahead), and made
  // ready: where the entry's bins for this block start in memory and how
  // many bytes from there are the row's, so that an entry costs the wave
  // three v_readlane and its loads, with immediate offsets.  An entry whose
  // first bin lies before the row's (`early`: the first blocks only) starts
  // at the row, and its lanes' offsets are formed whole.
  struct Meta {
    int32_t row, lag;
    double w, w2;
  };
  struct Ready {
    int64_t addr;
    int32_t bytes, w0;
    double w, w2;
    uint64_t ends, early;
  };
  auto load_meta = [&](int64_t e0) {
    const int64_t e = e0 + lane;
    const bool in = e < e_hi;
    const int64_t ec = in ? e : e_hi - 1;
    Meta m;
    m.row = a.rowid[ec];
    m.lag = in ? a.lag[ec] : kLagMask;  // past the end: no bins, no flag
    m.w = in ? w[ec] : 0.0;
    m.w2 = DS && in ? w2[ec] : 0.0;
    return m;
  };
  auto ready = [&](const Meta &m) {
    Ready x;
    const int n = min(m.lag & kLagMask, (int)T);
    x.w0 = t0 - n;
    const int skip = max(x.w0, 0), left = max(a.sp.Tp - skip, 0);
    x.addr = (int64_t)(a.prev + ((int64_t)m.row * B + b) * T + skip);
    x.bytes = n < t_end ? left * 4 : 0;
    x.w = m.w;
    x.w2 = m.w2;
    x.ends = __ballot((m.lag & kLastInGroup) != 0);
    x.early = __ballot(x.w0 < 0 && x.bytes != 0);
    return x;
  };
  auto fetch = [&](const Ready &m, int q, float (&v)[C][R]) {
    if ((m.early >> q & ((1ull << C) - 1ull)) == 0) {  // uniform
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const __amdgpu_buffer_rsrc_t rs =
            make_rsrc((const void *)readlane_i64(m.addr, q + c),
                      (uint32_t)__builtin_amdgcn_readlane(m.bytes, q + c));
#pragma unroll
        for (int r = 0; r < R; ++r)
          v[c][r] = buffer_load(rs, (uint32_t)lane * 4u + 256u * (uint32_t)r);
      }
      return;
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const __amdgpu_buffer_rsrc_t rs =
          make_rsrc((const void *)readlane_i64(m.addr, q + c),
                    (uint32_t)__builtin_amdgcn_readlane(m.bytes, q + c));
      const int w0 = min(__builtin_amdgcn_readlane(m.w0, q + c), 0);
#pragma unroll
      for (int r = 0; r < R; ++r)
        v[c][r] = buffer_load(rs, bin_offset(w0 + lane + 64 * r));
    }
  };
  // a group's sums to memory too, as the two-pass order stores them
  auto keep_sums = [&](int g, const double (&x)[R]) {
    const __amdgpu_buffer_rsrc_t os = make_rsrc(
        a.gsum + ((g0 + g) * B + b) * T, (uint32_t)a.sp.Tc * 4u);
#pragma unroll
    for (int r = 0; r < R; ++r)
      buffer_store((float)x[r], os, (uint32_t)(tl + 64 * r) * 4u);
  };
  auto consume = [&](const Ready &m, int q, const float (&v)[C][R]) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const double wk = readlane_f64(m.w, q + c);
      const double dk = DS ? readlane_f64(m.w2, q + c) : 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double x = (double)v[c][r];
        S[r] = fma(wk, x, S[r]);
        if (DS) Sd[DS ? r : 0] = fma(dk, x, Sd[DS ? r : 0]);
      }
      if (!one && (m.ends >> (q + c) & 1ull) != 0) {  // uniform
#pragma unroll
        for (int r = 0; r < R; ++r)
          gs[gl * TB + 64 * r + lane] = (float)S[r];
        if (a.gsum) keep_sums(gl, S);
#pragma unroll
        for (int r = 0; r < R; ++r) S[r] = 0.0;
        gl += 1;
      }
    }
  };
  if (e_hi > e_lo) {  // uniform
    Meta next = load_meta(e_lo);
    float va[C][R], vb[C][R];
    for (int64_t blk = e_lo; blk < e_hi; blk += 64) {
      const Ready cur = ready(next);
      next = load_meta(blk + 64);
      const int n = (int)min((int64_t)64, e_hi - blk);
      fetch(cur, 0, va);
      for (int q = 0; q < n; q += 2 * C) {
        if (q + C < n) fetch(cur, q + C, vb);
        consume(cur, q, va);
        if (q + C >= n) break;
        if (q + 2 * C < n) fetch(cur, q + 2 * C, va);
        consume(cur, q + C, vb);
      }
    }
  }
  if (DS || one) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      part[wave * TB + 64 * r + lane] = DS ? Sd[DS ? r : 0] : S[r];
  }
  if (!a.cur && !one) return;  // uniform
  __syncthreads();
  // the shared sum of a bin, in wave order, rounded as a group's sum is
  auto shared_sum = [&](int r) {
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < NW; ++q) sum += part[q * TB + 64 * r + lane];
    return (double)(float)sum;
  };

  if (one && a.gsum && ng && wave == 0) {
    double x[R];
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = shared_sum(r);
    keep_sums(0, x);
  }
  if (!a.cur) return;  // uniform

  // directions d0 .. d0+DW-1 and bin rows r0 .. r0+RW-1 of this wave
  constexpr int NWD = DP < NW ? DP : NW, DW = DP / NWD;
  constexpr int NWT = NW / NWD, RW = R < NWT ? 1 : R / NWT;
  const int d0 = wave % NWD * DW, r0 = wave / NWD * RW;
  if (r0 >= R) return;  // uniform
  double acc[DS ? 1 : DW][RW];
  if (!DS) {
#pragma unroll
    for (int d = 0; d < DW; ++d)
#pragma unroll
      for (int r = 0; r < RW; ++r) acc[DS ? 0 : d][r] = 0.0;
    // (the BRDF rows by LDS broadcast; by scalar loads 10 % slower)
#pragma unroll 4
    for (int g = 0; g < ng; ++g) {
      double x[RW];
#pragma unroll
      for (int r = 0; r < RW; ++r)
        x[r] = one ? shared_sum(r0 + r)
                   : (double)gs[g * TB + 64 * (r0 + r) + lane];
#pragma unroll
      for (int d = 0; d < DW; ++d) {
        const double cd = ct[g * DP + d0 + d];
#pragma unroll
        for (int r = 0; r < RW; ++r)
          acc[DS ? 0 : d][r] = fma(cd, x[r], acc[DS ? 0 : d][r]);
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[0][r] = shared_sum(r0 + r);
  }
  // the order's value: of the diffuse + specular plan the diffuse sum and
  // the direction's specular group, picked where it is written
  const int32_t *gmap =
      reinterpret_cast<const int32_t *>(part + (size_t)NW * TB);
  auto value = [&](int d, int r) {
    if (!DS) return acc[DS ? 0 : d][r];
    const int g = gmap[d0 + d];
    return (g >= 0 ? (double)gs[g * TB + 64 * (r0 + r) + lane] : 0.0) +
           acc[0][r];
  };
  const int64_t dstride = (int64_t)B * T;
  const int64_t base = j * D * dstride + (int64_t)b * T;
  const uint32_t span = (uint32_t)(((int64_t)(D - 1) * dstride + T) * 4);
  auto offset = [&](int d, int t, int end) {
    return d < D && t < end ? (uint32_t)((int64_t)d * dstride + t) * 4u
                            : kNoOffset;
  };
  const __amdgpu_buffer_rsrc_t rc =
      make_rsrc(a.cur + base, a.sp.last ? 0u : span);
  if (!a.tot_hi) {  // uniform
    const int nj = a.inj.n0 ? a.inj.n0[j] : -1;
#pragma unroll
    for (int d = 0; d < DW; ++d)
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const int t = tl + 64 * (r0 + r);
        double v = value(d, r);
        if (t == nj && d0 + d < D)
          v += a.inj.e0[(j * D + d0 + d) * B + b];
        buffer_store((float)v, rc, offset(d0 + d, t, a.sp.Tc));
      }
    return;
  }
  const __amdgpu_buffer_rsrc_t rh = make_rsrc(a.tot_hi + base, span);
  const __amdgpu_buffer_rsrc_t rl = make_rsrc(a.tot_lo + base, span);
  const __amdgpu_buffer_rsrc_t wl =
      make_rsrc(a.tot_lo + base, a.sp.last ? 0u : span);
  const __amdgpu_buffer_rsrc_t rp =
      make_rsrc((a.pair ? a.pair : a.cur) + base, a.pair ? span : 0u);
  constexpr int NP = DW * RW, KM = DS ? 16 : 8;  // (d, r) pairs
  constexpr int K = NP < KM ? NP : KM;           // loaded at a time
#pragma unroll
  for (int p0 = 0; p0 < NP; p0 += K) {
    float h[K], l[K], e[K];
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int d = d0 + (p0 + q) / RW, t = tl + 64 * (r0 + (p0 + q) % RW);
      h[q] = buffer_load(rh, offset(d, t, a.sp.Tv));
      l[q] = buffer_load(rl, offset(d, t, a.sp.Tv));
      e[q] = buffer_load(rp, offset(d, t, a.sp.Tp));
    }
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int d = (p0 + q) / RW, r = (p0 + q) % RW;
      const uint32_t off = offset(d0 + d, tl + 64 * (r0 + r), a.sp.Tc);
      const double x = value(d, r);
      const double v = a.sp.round ? (double)(float)x : x;
      double sum = (double)h[q] + (double)l[q];
      sum += (double)e[q];
      sum += v;
      const float hs = (float)sum;
      buffer_store((float)v, rc, off);
      buffer_store(hs, rh, off);
      buffer_store((float)(sum - (double)hs), wl, off);
    }
  }
}

template <int DP, int R, bool DS>
int launch_row_order(const spr_exchange_plan &p, RowArgs a, hipStream_t s) {
  const size_t lds = row_lds(p, R);
  a.n_tblk = (int)ceil_div(a.sp.Tc, 64 * R);
  a.nblocks = p.P * p.B * a.n_tblk;
  SPR_REQUIRE(a.nblocks <= max_blocks(64 * kRowWaves),
              "exchange grid too large");
  if (lds > 65536)
    SPR_HIP(hipFuncSetAttribute((const void *)row_order_kernel<DP, R, DS>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  hipLaunchKernelGGL((row_order_kernel<DP, R, DS>), dim3((unsigned)a.nblocks),
                     dim3(64 * kRowWaves), lds, s, a);
  SPR_LAUNCH_CHECK();
  return SPR_OK;
}

template <int R, bool DS>
int launch_dp(const spr_exchange_plan &p, const RowArgs &a, hipStream_t s) {
  switch (spr_padded_directions(p.D)) {
    case 1: return launch_row_order<1, R, DS>(p, a, s);
    case 2: return launch_row_order<2, R, DS>(p, a, s);
    case 4: return launch_row_order<4, R, DS>(p, a, s);
    case 8: return launch_row_order<8, R, DS>(p, a, s);
    case 16: return launch_row_order<16, R, DS>(p, a, s);
    case 32: return launch_row_order<32, R, DS>(p, a, s);
    case 64: return launch_row_order<64, R, DS>(p, a, s);
  }
  return fail(SPR_ERR_UNSUPPORTED, "row order: bad D");
}

}  // namespace

// The shape of an order: R bins per lane here, or 0 for the two passes.  The
// two costs are estimated in ns, fitted to 881 orders of shoeboxes of 42 to
// 1,170 patches, 1 to 64 directions, 1 to 8 bands, 100 to 4,000 bins (R = 1
// and 8 were tried too: at most 10 % faster anywhere):
// * here a workgroup costs 6 for its start, 0.2 per direction and bin row
//   written (0.13 with two weights), and per entry 0.06 (R = 4) or 0.048
//   (R = 2), 1.6 times that with two weights (an eighth of it per wave;
//   shared out over the chip), more where there are fewer groups than waves
//   (with one group they share it, and an entry costs 0.03 with R = 4: with
//   0.06 the two passes were taken for a 1,170-patch diffuse room, 3 bands,
//   700 bins: 612 us against 433);
// * a tile's workgroup (512 bins, or 256 with two weights) walks its entries
//   in 130 per merged entry and 12 per entry, whatever its bins; a workgroup
//   per CU runs at that pace, the chip takes 410 (530) in that time;
// * without tiles a workgroup (512 bins, or 2,048 with two weights) walks
//   its row in 900 per entry, at a rate of 0.2 (0.65) per entry;
// * two passes write and read the group sums, 0.0018 per group and bin, and
//   take a launch more, 8,000.
// Measured on 1,250 others (42 to 1,998 patches, 1, 2, 4, 8, 16, 24, 32 and 64
// directions, 100 to 3,000 bins) the choice is within 1.1 % of the best one on
// average with one weight and 0.7 % with two, at most 1.27 times slower
// (24 and 32 directions, one band: R = 2 would be better), and 1.55 and 1.29
// times faster than two passes.
int row_shape(const spr_exchange_plan &p, int64_t T, const OrderSpan &sp) {
  const int64_t DP = spr_padded_directions(p.D);
  if (p.order_shape < 0 || T >= ((int64_t)1 << 29) ||
      p.D * p.B * T >= ((int64_t)1 << 29))
    return 0;
  const bool ds = p.kind == SPR_PLAN_DS;
  // 64 directions at R = 4 keep 32 float64 sums per lane (with two weights,
  // none: one pick per direction)
  int R = p.order_shape ? (int)p.order_shape
                        : (DP <= 32 || ds) && sp.Tc > 128 ? 4 : 2;
  constexpr size_t kLds = 160 * 1024;
  if (!p.order_shape && row_lds(p, R) > kLds / 2) R = 2;
  const int64_t n = p.P * p.B, nb = n * ceil_div(sp.Tc, 64 * R);
  // (the two passes have half the threads or fewer for as many bins)
  if (row_lds(p, R) > kLds || nb > max_blocks(64 * kRowWaves)) return 0;
  if (p.order_shape) return R;
  const double E = (double)p.Vd / (double)p.P;
  const double groups = (double)(p.max_groups - (ds ? 1 : 0));
  const double idle = p.max_groups > 1 && groups < 8.0
                          ? std::pow(8.0 / std::max(groups, 1.0), 1.3)
                          : 1.0;
  const double here = (double)nb * (6.0 + (ds ? 0.13 : 0.2) * (double)(DP * R) +
                                    (R == 2            ? 0.048
                                     : p.max_groups > 1 ? 0.06
                                                        : 0.03) *
                                        (ds ? 1.6 : 1.0) * idle * E);
  double two = 8000.0 + (double)(n * sp.Tc) *
                            (0.0018 * (double)p.max_groups +
                             0.0033 * (double)DP);
  if (p.M) {
    const double tiles = (double)(p.tile_slots / p.tile_rows);
    const double blocks =
        tiles * (double)(p.B * ceil_div(sp.Tc, ds ? 256 : 512));
    two += (130.0 * (double)p.M + 12.0 * (double)p.Vd) / tiles *
           std::max(1.0, 0.55 + blocks / (ds ? 530.0 : 410.0));
  } else {
    const double blocks = (double)(n * ceil_div(sp.Tc, ds ? 2048 : 512));
    two += E * std::max(900.0, blocks * (ds ? 0.65 : 0.2));
  }
  return here < two ? R : 0;
}

int row_order(const spr_exchange_plan &p, int R, int64_t T, const float *prev,
              const float *pair, float *cur, float *tot_hi, float *tot_lo,
              float *gsum, const OrderStep &step, hipStream_t s) {
  RowArgs a{};
  a.D = (int)p.D;
  a.B = (int)p.B;
  a.T = (int)T;
  a.Vd = p.Vd;
  a.sp = step.span;
  a.inj = step.inj;
  a.max_groups = (int)p.max_groups;
  a.row_ptr = p.row_ptr;
  a.grp_ptr = p.grp_ptr;
  a.grp_start = p.grp_start;
  a.grp_key = p.grp_key;
  a.rowid = p.rowid;
  a.lag = p.lag;
  a.scal = p.scal;
  a.dscal = p.dscal;
  a.rtab = p.rtab;
  a.prev = prev;
  a.pair = pair;
  a.cur = cur;
  a.tot_hi = tot_hi;
  a.tot_lo = tot_lo;
  a.gsum = gsum;
  const bool ds = p.kind == SPR_PLAN_DS;
  switch (R) {
    case 2:
      return ds ? launch_dp<2, true>(p, a, s) : launch_dp<2, false>(p, a, s);
    case 4:
      return ds ? launch_dp<4, true>(p, a, s) : launch_dp<4, false>(p, a, s);
  }
  return fail(SPR_ERR_UNSUPPORTED, "spr_exchange_plan: order_shape is -1, 0, 2 or 4");
}

}  // namespace spr
