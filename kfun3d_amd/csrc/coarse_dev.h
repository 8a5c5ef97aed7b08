/*
 * coarse_dev.h -- the coarse levels' products in device code (coarse.hip,
 * jacobi.hip).
 */
#ifndef KF_COARSE_DEV_H
#define KF_COARSE_DEV_H

#include "kf_dev.h"

/* four values of a block row */
template <typename T>
struct cg_row { T v[4]; };

__device__ __forceinline__ cg_row<float> cg_ld(const float *p)
{
  const float4 t = *reinterpret_cast<const float4 *>(p);
  return {{t.x, t.y, t.z, t.w}};
}
__device__ __forceinline__ cg_row<double> cg_ld(const double *p)
{
  const double2 lo = reinterpret_cast<const double2 *>(p)[0], hi = reinterpret_cast<const double2 *>(p)[1];
  return {{lo.x, lo.y, hi.x, hi.y}};
}
__device__ __forceinline__ void cg_st(float *p, const cg_row<float> &r)
{
  *reinterpret_cast<float4 *>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
}
__device__ __forceinline__ void cg_st(double *p, const cg_row<double> &r)
{
  reinterpret_cast<double2 *>(p)[0] = make_double2(r.v[0], r.v[1]);
  reinterpret_cast<double2 *>(p)[1] = make_double2(r.v[2], r.v[3]);
}

/* a block row of A P as it is stored, and widened */
template <typename T>
struct cg_raw { cg_row<T> r; };
template <>
struct cg_raw<uint16_t> { uint2 r; };

template <typename T>
__device__ __forceinline__ void cg_ldraw(const T *p, cg_raw<T> &o) { o.r = cg_ld(p); }
__device__ __forceinline__ void cg_ldraw(const uint16_t *p, cg_raw<uint16_t> &o)
{
  o.r = *reinterpret_cast<const uint2 *>(p);
}
template <typename T>
__device__ __forceinline__ cg_row<double> cg_widen(const cg_raw<T> &o)
{
  return {{(double)o.r.v[0], (double)o.r.v[1], (double)o.r.v[2], (double)o.r.v[3]}};
}
__device__ __forceinline__ cg_row<double> cg_widen(const cg_raw<uint16_t> &o)
{
  return {{__uint_as_float(o.r.x << 16), __uint_as_float(o.r.x & 0xffff0000u), __uint_as_float(o.r.y << 16),
           __uint_as_float(o.r.y & 0xffff0000u)}};
}

/* lane I's value in each quad of lanes */
template <int I>
__device__ __forceinline__ double cg_quad(double v)
{
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), I * 0x55, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), I * 0x55, 0xf, 0xf, true));
}

#define AP_BATCH 8u   /* blocks of a row loaded together: all of them on a lattice */

/* up to AP_BATCH blocks of the row's n from the k0-th on, from place base on;
 * adds them to acc and moves base past the slice's */
template <typename TS>
__device__ __forceinline__ void ap_batch(const TS *__restrict__ ap, const uint32_t *__restrict__ apcol,
                                         const double *__restrict__ zc, uint32_t &base, uint32_t k0, uint32_t n,
                                         int c, double &acc)
{
  uint32_t at[AP_BATCH], kk[AP_BATCH];
#pragma unroll
  for (uint32_t k = 0; k < AP_BATCH; k++) {
    const uint64_t on = __ballot(k0 + k < n);
    const uint32_t below =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(on >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)on, 0u));
    /* whole quads are on or off: lane c has c more below it than its row */
    at[k] = k0 + k < n ? base + (below - (uint32_t)c) / 4u : base;
    base += (uint32_t)__popcll(on) / 4u;
  }
  cg_raw<TS> a[AP_BATCH];
  double z[AP_BATCH];   /* one component a lane */
#pragma unroll
  for (uint32_t k = 0; k < AP_BATCH; k++) kk[k] = apcol[at[k]];
#pragma unroll
  for (uint32_t k = 0; k < AP_BATCH; k++) cg_ldraw(ap + 16 * (size_t)at[k] + 4 * c, a[k]);
#pragma unroll
  for (uint32_t k = 0; k < AP_BATCH; k++) z[k] = zc[4 * (size_t)kk[k] + c];
#pragma unroll
  for (uint32_t k = 0; k < AP_BATCH; k++) {
    const cg_row<double> w = cg_widen(a[k]);
    double s = acc + w.v[0] * cg_quad<0>(z[k]);
    s = s + w.v[1] * cg_quad<1>(z[k]);
    s = s + w.v[2] * cg_quad<2>(z[k]);
    s = s + w.v[3] * cg_quad<3>(z[k]);
    acc = k0 + k < n ? s : acc;
  }
}

/* component c of row r of (A P) z_c: the A P blocks in ascending aggregate,
 * each component summed a[c][0] z0 + ... + a[c][3] z3 in FP64, the row's first
 * AP_BATCH blocks from ap1, the rest from ap */
template <typename TS, typename TA>
__device__ __forceinline__ double ap_product(uint32_t r, int c, const uint32_t *__restrict__ aprp,
                                             const uint32_t *__restrict__ apcol, const TA *__restrict__ ap,
                                             const TS *__restrict__ ap1, const double *__restrict__ zc)
{
  const uint32_t n = aprp[r + 1] - aprp[r];
  uint32_t base = aprp[r & ~15u];
  double acc = 0.0;
  ap_batch<TS>(ap1, apcol, zc, base, 0u, n, c, acc);
  for (uint32_t k0 = AP_BATCH; __any(k0 < n); k0 += AP_BATCH) ap_batch<TA>(ap, apcol, zc, base, k0, n, c, acc);
  return acc;
}

/* component c of aggregate I's sum over its members, ascending, eight at a
 * time loaded together (one by one, an index and its value were 8 round trips
 * of memory in a row) */
__device__ __forceinline__ double member_sum(uint32_t I, int c, const uint32_t *__restrict__ mptr,
                                             const uint32_t *__restrict__ mlist, const double *__restrict__ v)
{
  constexpr uint32_t MB = 8;
  const uint32_t m1 = mptr[I + 1];
  double s = 0.0;
  for (uint32_t m = mptr[I]; m < m1; m += MB) {
    uint32_t j[MB];
    double x[MB];
#pragma unroll
    for (uint32_t i = 0; i < MB; i++) j[i] = mlist[min(m + i, m1 - 1u)];
#pragma unroll
    for (uint32_t i = 0; i < MB; i++) x[i] = v[4 * (size_t)j[i] + c];
#pragma unroll
    for (uint32_t i = 0; i < MB; i++) s = m + i < m1 ? s + x[i] : s;
  }
  return s;
}

/* One level of the multilevel preconditioner below JAC_SMALL_ROWS rows, for
 * the launch that runs all of these (jacobi.hip): the level above hands it
 * its members' sums in b and takes x */
struct kf_small_level {
  uint32_t N, nslice;
  int K, sweeps;
  const uint32_t *rowptr, *col, *diag, *scol;
  const void *a, *val, *near;
  const uint32_t *mptr, *mlist;     /* members, of the level above */
  double *b, *x;
  /* towards the level below it (none: aprp is NULL) */
  const uint32_t *aprp, *apcol, *agg;
  const void *ap, *ap1;
  void *t;
};
#define KF_SMALL_LEVELS 8
struct kf_small_levels { kf_small_level l[KF_SMALL_LEVELS]; };

/* false: the context's solve is not one for that launch */
bool kf_jac_small_level(kf_ctx *c, kf_small_level *o);
void kf_jac_small_levels(kf_ctx *c, const kf_small_levels &s, int n, const double *b);

#endif
