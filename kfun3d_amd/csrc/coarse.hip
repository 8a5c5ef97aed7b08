/*
 * coarse.hip -- the two-level preconditioner (kf_options.coarse) on gfx950.
 *
 * The reference preconditions GMRES with block ILU(0) alone
 * (matrix/ilu.cpp:49-138, matrix/sptrsv.cpp:34-73).  Its Krylov count grows
 * with the mesh: the error modes that ILU(0) leaves are global.  This adds
 * a coarse level over aggregates of neighbouring vertices (host/aggregate.c):
 *   Ac = P^T A P                (Galerkin; P piecewise constant per component)
 *   z  = P Ac^-1 P^T b          (Ac^-1: block ILU(0) of Ac, the same kernels
 *                                as the fine level, in a matrix-only context,
 *                                solved exactly or by coarse_sweeps Jacobi
 *                                sweeps; with coarse = L > 1, the same scheme
 *                                again on Ac, L levels below the fine one)
 *   x  = z + (LU)^-1 (b - A z)  (the fine ILU(0) solve on the remainder,
 *                                exact or by jacobi_sweeps sweeps)
 * a fixed linear preconditioner, so plain left-preconditioned GMRES keeps
 * working.  A is the fill's Jacobian, read before the fine factorisation
 * overwrites it, and enters only as A P: the fine rows with their blocks
 * summed by the aggregate of their column (about 6 blocks a row on a
 * lattice, against 15 in A).  A P serves both the Galerkin product
 * (P^T (A P)) and the remainder b - (A P) z_c, so the full Jacobian is
 * neither kept nor re-read per application.  A P and the Galerkin sums are
 * FP64 with an FP64 preconditioner and FP32 otherwise; the coarse factors
 * take the fine level's precision (FP64, FP32, or BF16-stored with FP32
 * arithmetic).
 *
 * Kernels (a quad of lanes per block row, lane c forming component c, as
 * spmv.hip; workgroups remapped XCD by XCD):
 *   k_gather_sum   a block = the sum of listed blocks in ascending position:
 *                  A P from the fine blocks (with its BF16 copy, with a BF16
 *                  preconditioner), then P^T A P from A P
 *   k_restrict     coarse vector = sum of the aggregate's members, ascending
 *   k_coarse_resid t = b - (A P) z_c (FP32 where the fine solve is FP32
 *                  sweeps)
 *   k_prolong_add  x += P z_c (with Jacobi sweeps: inside their last sweep)
 * Every sum runs in a fixed order, so the preconditioner is deterministic.
 */
#include <cstring>

#include "coarse_dev.h"

#define CG_WG 256   /* 64 block rows per workgroup */

struct kf_coarse {
  kf_ctx *cc;          /* the coarse matrix: pattern, plans, values, factors */
  uint32_t nc;         /* aggregates */
  size_t cnnzb, nap;
  uint32_t *agg;       /* [N] aggregate of each fine vertex */
  uint32_t *mptr, *mlist;   /* members of each aggregate */
  uint32_t *aprp;      /* A P pattern: where a fine row's blocks would start row by row */
  uint32_t *appos, *apcol;      /* ... the place of each, and the aggregates by place */
  uint32_t *apgptr, *apglist;   /* fine block positions of each A P block */
  uint32_t *gptr, *glist;   /* A P places of each coarse block */
  double *ap64;        /* A P values by place (FP64 preconditioner) ... */
  float *ap32;         /* ... or FP32 */
  uint16_t *apbf;      /* ... and in BF16, for the remainder product with a BF16 preconditioner */
  double *rc, *zc;     /* coarse right-hand side and solution, 4 nc */
  double *t;           /* the fine remainder b - A z, 4 N */
  float *t32;          /* ... in FP32, where the fine solve is FP32 sweeps */
};

template <typename T>
static T *cupload(const T *h, size_t n)
{
  T *p = NULL;
  KF_CHECK(hipMalloc((void **)&p, (n ? n : 1) * sizeof(T)));
  if (n) KF_CHECK(hipMemcpy(p, h, n * sizeof(T), hipMemcpyHostToDevice));
  return p;
}

/* rounded to nearest even */
__device__ __forceinline__ uint32_t cg_bf16(float v)
{
  uint32_t u = __float_as_uint(v);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return u >> 16;
}

/* pos: where block b goes (NULL: to b); bf: the BF16 copy, or NULL.
 * The lists' blocks are loaded GB at a time, before their sums: A P of
 * 216x72x72 with its BF16 copy 0.36 ms (0.47 ms, and 0.34 ms for the copy,
 * with one block at a time and a kernel of its own). */
template <typename T>
__global__ __launch_bounds__(CG_WG) void k_gather_sum(uint32_t nb, const uint32_t *__restrict__ gptr,
                                                    const uint32_t *__restrict__ glist, const T *__restrict__ a,
                                                    T *__restrict__ ac, const uint32_t *__restrict__ pos,
                                                    uint16_t *__restrict__ bf)
{
  constexpr uint32_t GB = 4;
  const uint32_t b = kf_xcd_block() * (CG_WG / 4) + (threadIdx.x >> 2);
  const int c = threadIdx.x & 3;
  if (b >= nb) return;
  const uint32_t k1 = gptr[b + 1];
  const size_t at = pos ? pos[b] : b;
  cg_row<T> s = {{T(0), T(0), T(0), T(0)}};
  for (uint32_t k = gptr[b]; k < k1; k += GB) {
    uint32_t j[GB];
    cg_row<T> p[GB];
#pragma unroll
    for (uint32_t i = 0; i < GB; i++) j[i] = glist[min(k + i, k1 - 1u)];
#pragma unroll
    for (uint32_t i = 0; i < GB; i++) p[i] = cg_ld(a + 16 * (size_t)j[i] + 4 * c);
#pragma unroll
    for (uint32_t i = 0; i < GB; i++)
#pragma unroll
      for (int m = 0; m < 4; m++) s.v[m] = k + i < k1 ? s.v[m] + p[i].v[m] : s.v[m];
  }
  cg_st(ac + 16 * at + 4 * c, s);
  if constexpr (sizeof(T) == 4)
    if (bf)
      *reinterpret_cast<uint2 *>(bf + 16 * at + 4 * c) =
          make_uint2(cg_bf16(s.v[0]) | cg_bf16(s.v[1]) << 16, cg_bf16(s.v[2]) | cg_bf16(s.v[3]) << 16);
}

__global__ __launch_bounds__(CG_WG) void k_restrict(uint32_t nc, const uint32_t *__restrict__ mptr,
                                                    const uint32_t *__restrict__ mlist,
                                                    const double *__restrict__ v, double *__restrict__ rc)
{
  const uint32_t I = kf_xcd_block() * (CG_WG / 4) + (threadIdx.x >> 2);
  const int c = threadIdx.x & 3;
  if (I >= nc) return;
  rc[4 * (size_t)I + c] = member_sum(I, c, mptr, mlist, v);
}

/* ---- A P by places ------------------------------------------------------------
 *
 * A slice of 16 rows is a wavefront's: its blocks lie together, first all the
 * rows' first blocks, then the second ones of the rows that have one, and so
 * on, so that a load instruction reads one contiguous run and nothing is
 * padded (a lattice row has 5 or 8 A P blocks).  A wavefront finds its rows'
 * places by counting lanes: no index is loaded. */

/* the places of row by row positions, and the aggregates by place */
__global__ __launch_bounds__(CG_WG) void k_ap_places(uint32_t N, const uint32_t *__restrict__ aprp,
                                                     const uint32_t *__restrict__ col, uint32_t *__restrict__ pos,
                                                     uint32_t *__restrict__ pcol)
{
  const uint32_t r = blockIdx.x * CG_WG + threadIdx.x;
  if (r >= N) return;
  const uint32_t r0 = r & ~15u, r1 = min(r0 + 16u, N), j0 = aprp[r], n = aprp[r + 1] - j0;
  for (uint32_t k = 0; k < n; k++) {
    uint32_t at = aprp[r0];
    for (uint32_t i = r0; i < r1; i++) {
      const uint32_t m = aprp[i + 1] - aprp[i];
      at += min(m, k) + (i < r && m > k ? 1u : 0u);
    }
    pos[j0 + k] = at;
    pcol[at] = col[j0 + k];
  }
}

__global__ __launch_bounds__(CG_WG) void k_ap_relist(uint32_t n, const uint32_t *__restrict__ pos,
                                                     uint32_t *__restrict__ list)
{
  const uint32_t i = blockIdx.x * CG_WG + threadIdx.x;
  if (i < n) list[i] = pos[list[i]];
}

/* t = b - (A P) z_c; per row the A P blocks in ascending aggregate, each
 * component summed a[c][0] z0 + ... + a[c][3] z3 in FP64, the row's first
 * AP_BATCH blocks from ap1 (BF16 with a BF16 preconditioner, else ap itself),
 * the rest from ap; stored as TT (float where the fine sweeps round it to
 * FP32 on reading anyway).  Bound by memory: 288x96x96 in BF16 0.224 -> 0.170 ms
 * (before: 8 padded slots a row, a quad loading each z four times over, 112
 * VGPRs; the compact copy alone left it at 0.224). */
template <typename TS, typename TA, typename TT>
__global__ __launch_bounds__(CG_WG) void k_coarse_resid(uint32_t N, const uint32_t *__restrict__ aprp,
                                                        const uint32_t *__restrict__ apcol,
                                                        const TA *__restrict__ ap, const TS *__restrict__ ap1,
                                                        const double *__restrict__ zc,
                                                        const double *__restrict__ b, TT *__restrict__ t)
{
  const uint32_t r = kf_xcd_block() * (CG_WG / 4) + (threadIdx.x >> 2);
  const int c = threadIdx.x & 3;
  if (r >= N) return;
  const double acc = ap_product<TS, TA>(r, c, aprp, apcol, ap, ap1, zc);
  const size_t o = 4 * (size_t)r + c;
  t[o] = (TT)(b[o] - acc);
}

__global__ __launch_bounds__(CG_WG) void k_prolong_add(size_t n4, const uint32_t *__restrict__ agg,
                                                       const double *__restrict__ zc, double *__restrict__ x)
{
  const size_t i = (size_t)blockIdx.x * CG_WG + threadIdx.x;
  if (i < n4) x[i] = x[i] + zc[4 * (size_t)agg[i >> 2] + (i & 3)];
}

/* the coarse level, built on first use from the context's own pattern */
static kf_coarse *coarse_build(kf_ctx *c)
{
  const size_t N = c->d.N, nnzb = c->nnzb;
  kf_prep fp;
  memset(&fp, 0, sizeof(fp));
  fp.N = N;
  fp.nnzb = nnzb;
  fp.rowptr = (uint32_t *)kf_xmalloc((N + 1) * sizeof(uint32_t));
  fp.col = (uint32_t *)kf_xmalloc((nnzb + 1) * sizeof(uint32_t));
  fp.diag = (uint32_t *)kf_xmalloc((N + 1) * sizeof(uint32_t));
  KF_CHECK(hipMemcpy(fp.rowptr, c->d.rowptr, (N + 1) * sizeof(uint32_t), hipMemcpyDeviceToHost));
  KF_CHECK(hipMemcpy(fp.col, c->d.col, nnzb * sizeof(uint32_t), hipMemcpyDeviceToHost));
  KF_CHECK(hipMemcpy(fp.diag, c->d.diag, N * sizeof(uint32_t), hipMemcpyDeviceToHost));
  kf_coarse_host h;
  kf_build_coarse(&fp, &h);
  free(fp.rowptr);
  free(fp.col);
  free(fp.diag);

  kf_options co = c->opt;
  co.prec = c->opt.prec;
  co.ilu_exact = 0;
  co.jacobi_sweeps = c->opt.coarse_sweeps;   /* the coarse levels' own solves */
  co.coarse = c->opt.coarse - 1;   /* further levels below this one */
  kf_coarse *k = new kf_coarse();
  k->cc = kf_ctx_create_matrix(&h.prep, &co, c);
  k->nc = (uint32_t)h.prep.N;
  k->cnnzb = h.prep.nnzb;
  k->nap = h.nap;
  k->agg = cupload(h.agg, N);
  k->mptr = cupload(h.mptr, (size_t)k->nc + 1);
  k->mlist = cupload(h.mlist, N);
  k->aprp = cupload(h.aprp, N + 1);
  uint32_t *col = cupload(h.apcol, h.nap);
  /* one block more than there is, for lanes without one */
  KF_CHECK(hipMalloc((void **)&k->appos, (h.nap + 1) * sizeof(uint32_t)));
  KF_CHECK(hipMalloc((void **)&k->apcol, (h.nap + 1) * sizeof(uint32_t)));
  KF_CHECK(hipMemset(k->apcol + h.nap, 0, sizeof(uint32_t)));
  k->apgptr = cupload(h.apgptr, h.nap + 1);
  k->apglist = cupload(h.apglist, nnzb);
  k->gptr = cupload(h.gptr, k->cnnzb + 1);
  k->glist = cupload(h.glist, h.nap);
  hipLaunchKernelGGL(k_ap_places, dim3(kf_blocks_for(N, CG_WG)), dim3(CG_WG), 0, c->stream, (uint32_t)N, k->aprp, col,
                     k->appos, k->apcol);
  KF_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_ap_relist, dim3(kf_blocks_for(h.nap, CG_WG)), dim3(CG_WG), 0, c->stream, (uint32_t)h.nap,
                     k->appos, k->glist);
  KF_LAUNCH_CHECK();
  KF_CHECK(hipStreamSynchronize(c->stream));
  KF_CHECK(hipFree(col));
  KF_CHECK(hipMalloc((void **)&k->rc, 4 * (size_t)k->nc * sizeof(double)));
  KF_CHECK(hipMalloc((void **)&k->zc, 4 * (size_t)k->nc * sizeof(double)));
  KF_CHECK(hipMalloc((void **)&k->t, 4 * N * sizeof(double)));
  kf_free_coarse(&h);
  return k;
}

/* P^T (A P) from A P into a coarse value array */
template <typename T>
static void galerkin_from_ap(kf_ctx *c, const kf_coarse *k, const T *ap, T *out)
{
  hipLaunchKernelGGL(k_gather_sum<T>, dim3(kf_blocks_for(k->cnnzb, CG_WG / 4)), dim3(CG_WG), 0, c->stream,
                     (uint32_t)k->cnnzb, k->gptr, k->glist, ap, out, (const uint32_t *)NULL, (uint16_t *)NULL);
  KF_LAUNCH_CHECK();
}

/* A P from the fill's values (before the fine factorisation overwrites
 * them), then P^T A P into the coarse context and its ILU(0) */
void kf_coarse_factor(kf_ctx *c)
{
  if (!c->coarse) c->coarse = coarse_build(c);
  kf_coarse *k = (kf_coarse *)c->coarse;
  kf_ctx *cc = k->cc;
  const bool f64 = c->opt.prec == KF_PREC_FP64, bf = c->opt.prec == KF_PREC_BF16;
  cc->opt.prec = c->opt.prec;   /* the coarse factors follow the fine level's precision */
  cc->opt.jacobi_sweeps = cc->opt.coarse_sweeps = c->opt.coarse_sweeps;
  if (cc->opt.coarse != c->opt.coarse - 1) {   /* the number of levels changed */
    if (c->opt.coarse == 1) kf_coarse_destroy(cc);
    cc->opt.coarse = c->opt.coarse - 1;
  }
  if (f64 ? k->ap32 != NULL : k->ap64 != NULL) {
    /* the precision changed: drop the other copy of A P (its last reader is
     * done once the stream is), so that a stale one is never read */
    KF_CHECK(hipStreamSynchronize(c->stream));
    KF_CHECK(hipFree(f64 ? (void *)k->ap32 : (void *)k->ap64));
    if (f64) k->ap32 = NULL;
    else k->ap64 = NULL;
  }
  const int s = kf_prof_begin(c, KP_COARSE_FACTOR);
  const uint32_t nb = kf_blocks_for(k->nap, CG_WG / 4);
  if (f64) {
    if (!k->ap64) KF_CHECK(hipMalloc((void **)&k->ap64, 16 * (k->nap + 1) * sizeof(double)));
    hipLaunchKernelGGL(k_gather_sum<double>, dim3(nb), dim3(CG_WG), 0, c->stream, (uint32_t)k->nap, k->apgptr,
                       k->apglist, (const double *)c->a64, k->ap64, k->appos, (uint16_t *)NULL);
    KF_LAUNCH_CHECK();
    galerkin_from_ap<double>(c, k, k->ap64, cc->a64);
  } else {
    if (!c->a32) {
      fprintf(stderr, "kf: two-level preconditioner: no single-precision Jacobian (ComputeA must run first)\n");
      abort();
    }
    if (!k->ap32) KF_CHECK(hipMalloc((void **)&k->ap32, 16 * (k->nap + 1) * sizeof(float)));
    if (bf && !k->apbf) KF_CHECK(hipMalloc((void **)&k->apbf, 16 * (k->nap + 1) * sizeof(uint16_t)));
    if (!cc->a32) KF_CHECK(hipMalloc((void **)&cc->a32, 16 * k->cnnzb * sizeof(float)));
    hipLaunchKernelGGL(k_gather_sum<float>, dim3(nb), dim3(CG_WG), 0, c->stream, (uint32_t)k->nap, k->apgptr,
                       k->apglist, (const float *)c->a32, k->ap32, k->appos, bf ? k->apbf : (uint16_t *)NULL);
    KF_LAUNCH_CHECK();
    galerkin_from_ap<float>(c, k, k->ap32, cc->a32);
  }
  if (cc->opt.coarse) kf_coarse_factor(cc);   /* the next level, from the Galerkin values */
  kf_launch_ilu(cc);
  kf_prof_end(c, s);
}

/* The levels below c in one launch, from the members' sums of b to k->zc,
 * where they are small enough for it (false: they are not, nothing launched) */
static bool small_levels(kf_ctx *c, const kf_coarse *k, const double *b)
{
  kf_small_levels s;
  int n = 0;
  for (;;) {
    kf_ctx *cc = k->cc;
    if (n == KF_SMALL_LEVELS) return false;
    kf_small_level &l = s.l[n++];
    memset(&l, 0, sizeof(l));
    if (cc->opt.prec != c->opt.prec || !kf_jac_small_level(cc, &l)) return false;
    l.mptr = k->mptr;
    l.mlist = k->mlist;
    l.b = k->rc;
    l.x = k->zc;
    if (!cc->opt.coarse) break;
    kf_coarse *kk = (kf_coarse *)cc->coarse;
    const bool f64 = c->opt.prec == KF_PREC_FP64, bf = c->opt.prec == KF_PREC_BF16;
    if (!kk || (f64 ? !kk->ap64 : !kk->ap32) || (bf && !kk->apbf)) return false;
    if (!f64 && !kk->t32) KF_CHECK(hipMalloc((void **)&kk->t32, 4 * (size_t)cc->d.N * sizeof(float)));
    l.aprp = kk->aprp;
    l.apcol = kk->apcol;
    l.agg = kk->agg;
    l.ap = f64 ? (const void *)kk->ap64 : (const void *)kk->ap32;
    l.ap1 = bf ? (const void *)kk->apbf : l.ap;
    l.t = f64 ? (void *)kk->t : (void *)kk->t32;
    k = kk;
  }
  kf_jac_small_levels(c, s, n, b);
  return true;
}

/* x = M b with the two-level preconditioner (b, x device, 4N, not aliased) */
void kf_coarse_apply(kf_ctx *c, const double *b, double *x)
{
  kf_coarse *k = (kf_coarse *)c->coarse;
  if (!k) {
    fprintf(stderr, "kf: two-level preconditioner: ComputeNumericalILU has not run with coarse = 1\n");
    abort();
  }
  const bool f64 = c->opt.prec == KF_PREC_FP64, bf = c->opt.prec == KF_PREC_BF16;
  if ((f64 ? !k->ap64 : !k->ap32) || (bf && !k->apbf)) {
    fprintf(stderr, "kf: two-level preconditioner: the preconditioner's precision changed since "
                    "ComputeNumericalILU\n");
    abort();
  }
  kf_check_aligned(b, "b");
  kf_check_aligned(x, "x");
  const kf_dv &d = c->d;
  const int s = kf_prof_begin(c, KP_COARSE);
  if (!small_levels(c, k, b)) {
    hipLaunchKernelGGL(k_restrict, dim3(kf_blocks_for(k->nc, CG_WG / 4)), dim3(CG_WG), 0, c->stream, k->nc, k->mptr,
                       k->mlist, b, k->rc);
    KF_LAUNCH_CHECK();
    if (k->cc->opt.coarse) kf_coarse_apply(k->cc, k->rc, k->zc);   /* the coarse system by the same scheme */
    else if (k->cc->opt.jacobi_sweeps > 0) kf_launch_jacobi(k->cc, k->rc, k->zc);
    else kf_launch_sptrsv(k->cc, k->rc, k->zc, NULL);
  }
  const uint32_t nb = kf_blocks_for(d.N, CG_WG / 4);
  const size_t n4 = 4 * (size_t)d.N;
  const bool sweeps = c->opt.jacobi_sweeps > 0;
  const bool t32 = sweeps && !f64;
  if (t32 && !k->t32) KF_CHECK(hipMalloc((void **)&k->t32, n4 * sizeof(float)));
#define CG_RESID(TS, TA, TT, ap, ap1, t)                                                                            \
  hipLaunchKernelGGL((k_coarse_resid<TS, TA, TT>), dim3(nb), dim3(CG_WG), 0, c->stream, d.N, k->aprp, k->apcol,      \
                     (const TA *)(ap), (const TS *)(ap1), k->zc, b, t)
  if (f64) CG_RESID(double, double, double, k->ap64, k->ap64, k->t);
  else if (bf && t32) CG_RESID(uint16_t, float, float, k->ap32, k->apbf, k->t32);
  else if (bf) CG_RESID(uint16_t, float, double, k->ap32, k->apbf, k->t);
  else if (t32) CG_RESID(float, float, float, k->ap32, k->ap32, k->t32);
  else CG_RESID(float, float, double, k->ap32, k->ap32, k->t);
#undef CG_RESID
  KF_LAUNCH_CHECK();
  kf_prof_end(c, s);
  if (sweeps) {
    /* the fine solve by sweeps, x += P z_c in its last sweep */
    kf_launch_jacobi_ml(c, f64 ? (const void *)k->t : (const void *)k->t32, x, k->agg, k->zc);
    return;
  }
  kf_launch_sptrsv(c, k->t, x, NULL);
  hipLaunchKernelGGL(k_prolong_add, dim3(kf_blocks_for(n4, CG_WG)), dim3(CG_WG), 0, c->stream, n4, k->agg, k->zc, x);
  KF_LAUNCH_CHECK();
}

void kf_coarse_destroy(kf_ctx *c)
{
  kf_coarse *k = (kf_coarse *)c->coarse;
  if (!k) return;
  kf_coarse_destroy(k->cc);
  kf_ctx_destroy_matrix(k->cc);
  void *ptrs[] = {k->agg, k->mptr, k->mlist, k->aprp, k->appos, k->apcol, k->apgptr, k->apglist, k->gptr, k->glist,
                  k->ap64, k->ap32, k->apbf, k->rc, k->zc, k->t, k->t32};
  for (size_t i = 0; i < sizeof(ptrs) / sizeof(ptrs[0]); i++)
    if (ptrs[i]) KF_CHECK(hipFree(ptrs[i]));
  delete k;
  c->coarse = NULL;
}

/* the coarse level's size, its aggregate map and its Galerkin blocks (for
 * tests): returns the number of aggregates; with non-NULL arrays also copies
 * agg [N], the coarse pattern rowptr [nc + 1], col [cnnzb] and the blocks
 * [16 cnnzb] as the last factorisation formed them (before their ILU) */
extern "C" size_t kf_coarse_matrix(const GEOMETRY *g, size_t *cnnzb, unsigned *agg, unsigned *rowptr, unsigned *col,
                                   double *blocks)
{
  kf_ctx *c = kf_ctx_of(g);
  kf_coarse *k = (kf_coarse *)c->coarse;
  if (!k) return 0;
  KF_CHECK(hipStreamSynchronize(c->stream));
  if (cnnzb) *cnnzb = k->cnnzb;
  if (agg) KF_CHECK(hipMemcpy(agg, k->agg, (size_t)c->d.N * sizeof(uint32_t), hipMemcpyDeviceToHost));
  if (rowptr) KF_CHECK(hipMemcpy(rowptr, k->cc->d.rowptr, ((size_t)k->nc + 1) * sizeof(uint32_t), hipMemcpyDeviceToHost));
  if (col) KF_CHECK(hipMemcpy(col, k->cc->d.col, k->cnnzb * sizeof(uint32_t), hipMemcpyDeviceToHost));
  if (blocks) {
    /* the Galerkin product again from A P (the coarse values were factored
     * in place), into the host array */
    const size_t n = 16 * k->cnnzb;
    const bool f64 = c->opt.prec == KF_PREC_FP64;
    if (f64 ? !k->ap64 : !k->ap32) {
      fprintf(stderr, "kf: kf_coarse_matrix: the preconditioner's precision changed since ComputeNumericalILU\n");
      abort();
    }
    void *tmp = NULL;
    KF_CHECK(hipMalloc(&tmp, n * (f64 ? sizeof(double) : sizeof(float))));
    if (f64) galerkin_from_ap<double>(c, k, k->ap64, (double *)tmp);
    else galerkin_from_ap<float>(c, k, k->ap32, (float *)tmp);
    KF_CHECK(hipStreamSynchronize(c->stream));
    if (f64) {
      KF_CHECK(hipMemcpy(blocks, tmp, n * sizeof(double), hipMemcpyDeviceToHost));
    } else {
      float *h = (float *)kf_xmalloc(n * sizeof(float));
      KF_CHECK(hipMemcpy(h, tmp, n * sizeof(float), hipMemcpyDeviceToHost));
      for (size_t i = 0; i < n; i++) blocks[i] = (double)h[i];
      free(h);
    }
    KF_CHECK(hipFree(tmp));
  }
  return k->nc;
}
