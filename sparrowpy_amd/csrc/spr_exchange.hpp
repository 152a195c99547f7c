// Exchange plan conventions and buffer-descriptor helpers shared by the
// forward (exchange.hip) and adjoint (adjoint.hip) passes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "spr_common.hpp"

namespace spr {

// Entry metadata of the grouped plan: the delay word carries, in bit 30,
// the flag "last entry of its group" (delays are clamped below 2^30).
constexpr int32_t kLastInGroup = 0x40000000;
constexpr int32_t kLagMask = 0x3fffffff;

// Tile order of the grouped passes: destination fastest, then time block,
// then band.  With the XCD-contiguous block mapping, the blocks resident on
// one XCD at a time are neighbouring destinations (neighbouring patches of
// a wall) in the same band and time window, which read nearly the same
// source histogram segments -- so those reads are shared through L2/MALL.
__device__ __forceinline__ void dest_major_tile(uint32_t tile,
                                                int64_t nblocks, int B,
                                                int n_tblk, int64_t &j,
                                                int &b, int &tb) {
  const uint32_t nt = (uint32_t)n_tblk;
  const uint32_t P = (uint32_t)nblocks / ((uint32_t)B * nt);
  const uint32_t rest = tile / P;
  j = tile % P;
  tb = (int)(rest % nt);
  b = (int)(rest / nt);
}

// Time-major: consecutive tiles are the time blocks of one destination.
__device__ __forceinline__ void time_major_tile(uint32_t tile,
                                                int64_t nblocks, int B,
                                                int n_tblk, int64_t &j,
                                                int &b, int &tb) {
  const uint32_t nt = (uint32_t)n_tblk;
  const uint32_t P = (uint32_t)nblocks / ((uint32_t)B * nt);
  const uint32_t jb = tile / nt;
  tb = (int)(tile % nt);
  j = jb % P;
  b = (int)(jb / P);
}

// Raw buffer access with a gfx9 buffer descriptor: a load whose byte
// offset lies outside [0, bytes) returns 0 and a store there is dropped,
// with no branch and no memory access.  This lets every lane issue its
// loads unconditionally, so the compiler can count them and keep the next
// chunk's loads in flight while the current chunk is summed.
constexpr int kBufferWord3 = 0x00020000;   // gfx9 descriptor word 3
constexpr uint32_t kNoOffset = 0x80000000u;  // beyond every range used here

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p,
                                                            uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0,
                                           (int)bytes, kBufferWord3);
}

// Byte offset 4k of bin k of a row, kept whole.  For k < 0 the wrapped
// 32-bit value lies beyond every buffer used here and the load reads 0 --
// but only if the instruction receives it as computed: the compiler would
// otherwise move constant parts of the offset into the instruction's
// immediate field, and the hardware does not range-check the wrapped
// register offset plus that immediate as the 32-bit sum it stands for
// (loads of a row's first bins through such a pair return 0).  The empty
// asm makes the value opaque, so it is never split.
__device__ __forceinline__ uint32_t bin_offset(int k) {
  uint32_t off = (uint32_t)k * 4u;
  asm("" : "+v"(off));
  return off;
}

__device__ __forceinline__ float buffer_load(__amdgpu_buffer_rsrc_t r,
                                             uint32_t off) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}

__device__ __forceinline__ void buffer_store(float v,
                                             __amdgpu_buffer_rsrc_t r,
                                             uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r,
                                        (int)off, 0, 0);
}

__device__ __forceinline__ int64_t readlane_i64(int64_t u, int k) {
  const int32_t lo = __builtin_amdgcn_readlane((int32_t)u, k);
  const int32_t hi = __builtin_amdgcn_readlane((int32_t)(u >> 32), k);
  return ((int64_t)hi << 32) | (int64_t)(uint32_t)lo;
}
__device__ __forceinline__ double readlane_f64(double v, int k) {
  return __builtin_bit_cast(double,
                            readlane_i64(__builtin_bit_cast(int64_t, v), k));
}

// BRDF row of entry e (source i -> destination j): brdf_index[w_i] * S +
// s_ij (0 without a BRDF).
__device__ __forceinline__ int64_t entry_brdf_row(
    int64_t i, int64_t j, const double *__restrict__ centers,
    const int64_t *__restrict__ wall_ids, int64_t S,
    const int64_t *__restrict__ brdf_index,
    const double *__restrict__ in_dirs) {
  if (!in_dirs) return 0;
  d3 u = load3(centers + 3 * i) - load3(centers + 3 * j);
  u = div(u, norm(u));
  const int64_t w = wall_ids[i];
  return brdf_index[w] * S + nearest_direction(in_dirs + w * S * 3, S, u);
}

// The bins of one order that can hold energy: bins of the source histograms
// from Tp on, of the result from Tc on and of the total so far from Tv on
// are 0 and are neither read nor written.  Of the last order only the total
// is kept, rounded; round adds the order to the total as rounded to float32
// (as when it is read back from its histogram).
struct OrderSpan {
  int Tp, Tc, Tv;
  int last, round;
};
// Energy injected into every order of the running sum x_{k+1} = x_0 + A x_k
// (spr_exchange_sum): one bin n0[i] per patch.
struct Injection {
  const double *e0 = nullptr;   // [P, D, B]
  const int32_t *n0 = nullptr;  // [P]
};
struct OrderStep {
  OrderSpan span;
  Injection inj;
};
inline OrderSpan span_of(const OrderStep *step, int64_t T) {
  return step ? step->span : OrderSpan{(int)T, (int)T, (int)T, 0, 0};
}

// The passes of an order (exchange.hip, tiles.hip): the group sums row by
// row or on destination tiles, the spread over the directions, and the
// per-pair order.
int gather_rows(const spr_exchange_plan &p, int64_t T, const float *prev,
                float *gsum, const OrderStep &step, hipStream_t s);
int gather_tiles(const spr_exchange_plan &p, int64_t T, const float *prev,
                 float *gsum, const OrderStep &step, hipStream_t s);
int spread_rows(const spr_exchange_plan &p, int64_t T, const float *gsum,
                const float *prev, float *cur, float *tot_hi, float *tot_lo,
                const OrderStep &step, hipStream_t s);
// A whole order of a grouped or diffuse + specular plan in one launch
// (rows.hip) at R bins per lane, and the R to take (0: the two passes).
int row_shape(const spr_exchange_plan &p, int64_t T, const OrderSpan &sp);
int row_order(const spr_exchange_plan &p, int R, int64_t T, const float *prev,
              const float *pair, float *cur, float *tot_hi, float *tot_lo,
              float *gsum, const OrderStep &step, hipStream_t s);
int step_pairs(int64_t P, int64_t D, int64_t B, int64_t T,
               const int64_t *row_ptr, const int32_t *src, const int32_t *lag,
               const int32_t *dir, const double *coef, const float *prev,
               float *cur, float *tot_hi, float *tot_lo, const OrderStep *step,
               hipStream_t s);

// spr_exchange_orders on n_states order buffers taken in turn (sums.hip).
int exchange_orders(const char *name, const spr_exchange_plan &p, int64_t T,
                    int64_t K, int64_t reach, const double *e0dir,
                    const double *d0, double c, double dt, float *out,
                    float *lo, float *const *states, int64_t n_states,
                    float *gsum, int32_t *n0, int *err_flag, hipStream_t s);

// The passes of a backward order (adjoint.hip) on the bins below Tk that
// E_k can hold energy in, and below Tn for E_{k+1}.
int direction_sum(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
                  const float *mu, float *musum, hipStream_t s);
int adjoint_ds(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tk,
               int64_t Tn, int64_t Vd, const int64_t *tgptr,
               const int32_t *tkey, const int32_t *tlag, const int32_t *tm,
               const double *twa, const double *twc, const float *lam,
               const float *musum, const float *munext, const float *ek,
               float *muout, double *ga, hipStream_t s);
int spread_adjoint(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
                   const int64_t *grp_ptr, const int32_t *grp_key,
                   const double *rtab, const float *mu, float *nu,
                   hipStream_t s);
int table_grad(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tn,
               const int64_t *grp_ptr, const float *mu, const float *gsum,
               double *gg, hipStream_t s);
int gather_adjoint(int64_t P, int64_t D, int64_t B, int64_t T, int64_t Tk,
                   int64_t Tn, int64_t Vd, const int64_t *trow_ptr,
                   const int32_t *tgrp, const int32_t *tlag,
                   const double *tscal, const float *nu, const float *lam,
                   float *muout, hipStream_t s);

}  // namespace spr
