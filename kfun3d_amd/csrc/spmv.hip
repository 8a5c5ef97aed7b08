/*
 * spmv.hip -- y = A x with the assembled block Jacobian (BSR 4x4, the
 * pattern of matrix/init.cpp:7-74, the values of ComputeA / src/fill.c) on
 * gfx950.
 *
 * The reference never multiplies by its assembled matrix: its Krylov
 * operator is the matrix-free finite-difference product (src/kernel.c:24-45)
 * and A only feeds the ILU preconditioner.  This product serves the
 * first-order-operator mode of GMRES (kf_options.bsr_operator) and tools.
 *
 * Layout and order.  A quad of lanes owns one block row; lane c forms
 * component c:  y[4r + c] = sum over the row's blocks j in ascending column
 * of  a_j[c][0] x0 + a_j[c][1] x1 + a_j[c][2] x2 + a_j[c][3] x3,  each
 * product added to the running sum in that order, in FP64 (FP32-stored
 * values are widened first).  The four lanes of a quad read a block row by
 * row, so a wave's loads are whole blocks.  FP64: two blocks in flight, the
 * column's whole vector in each lane.  FP32: eight blocks in flight, of the
 * column's four x values each lane loads one and the quad exchanges them
 * (there 4 to 8 blocks in flight and 4 to 8 wavefronts a SIMD measure the
 * same).  Workgroups are remapped XCD by XCD (kf_xcd_block) so that each XCD
 * works on a contiguous slab of rows and its x gathers stay in its L2.  Bytes
 * per launch: nnzb (16 s + 4) + 64 N with s the stored value size (HBM-bound).
 */
#include "kf_dev.h"

#define SPMV_WG 256   /* 64 rows per workgroup */

/* a block row as it is stored */
template <typename T>
struct spmv_row;
template <>
struct spmv_row<double> {
  double2 u, v;
  __device__ __forceinline__ void load(const double *p)
  {
    u = reinterpret_cast<const double2 *>(p)[0];
    v = reinterpret_cast<const double2 *>(p)[1];
  }
  __device__ __forceinline__ void get(double a[4]) const { a[0] = u.x; a[1] = u.y; a[2] = v.x; a[3] = v.y; }
};
template <>
struct spmv_row<float> {
  float4 u;
  __device__ __forceinline__ void load(const float *p) { u = *reinterpret_cast<const float4 *>(p); }
  __device__ __forceinline__ void get(double a[4]) const
  {
    a[0] = (double)u.x; a[1] = (double)u.y; a[2] = (double)u.z; a[3] = (double)u.w;
  }
};

/* lane I's value in each quad of lanes */
template <int I>
__device__ __forceinline__ double spmv_quad(double v)
{
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), I * 0x55, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), I * 0x55, 0xf, 0xf, true));
}

template <typename T>
__global__ __launch_bounds__(SPMV_WG, 6) void k_bsr_spmv(uint32_t N, const uint32_t *__restrict__ rowptr,
                                                      const uint32_t *__restrict__ col, const T *__restrict__ a,
                                                      const double *__restrict__ x, double *__restrict__ y)
{
  const uint32_t r = kf_xcd_block() * (SPMV_WG / 4) + (threadIdx.x >> 2);
  const int c = threadIdx.x & 3;
  if (r >= N) return;   /* whole quads leave together */
  const uint32_t j1 = rowptr[r + 1];
  double acc = 0.0;
  uint32_t j = rowptr[r];
  if constexpr (sizeof(T) == 8) {
    /* two blocks at a time, the column's whole vector in each lane: a block of
     * FP64 is a line by itself and the product at the memory's rate (288x96x96
     * 1.04 ms; 1.08 with the exchange below, four blocks at a time) */
    for (; j + 1 < j1; j += 2) {
      const uint32_t k0 = col[j], k1 = col[j + 1];
      spmv_row<T> m0, m1;
      m0.load(a + 16 * (size_t)j + 4 * c);
      m1.load(a + 16 * (size_t)(j + 1) + 4 * c);
      const double4 u = *reinterpret_cast<const double4 *>(x + 4 * (size_t)k0);
      const double4 v = *reinterpret_cast<const double4 *>(x + 4 * (size_t)k1);
      double p[4], q[4];
      m0.get(p);
      m1.get(q);
      acc = acc + p[0] * u.x; acc = acc + p[1] * u.y; acc = acc + p[2] * u.z; acc = acc + p[3] * u.w;
      acc = acc + q[0] * v.x; acc = acc + q[1] * v.y; acc = acc + q[2] * v.z; acc = acc + q[3] * v.w;
    }
    if (j < j1) {
      spmv_row<T> m0;
      m0.load(a + 16 * (size_t)j + 4 * c);
      const double4 u = *reinterpret_cast<const double4 *>(x + 4 * (size_t)col[j]);
      double p[4];
      m0.get(p);
      acc = acc + p[0] * u.x; acc = acc + p[1] * u.y; acc = acc + p[2] * u.z; acc = acc + p[3] * u.w;
    }
    y[4 * (size_t)r + c] = acc;
    return;
  }
  constexpr uint32_t B = 8;   /* blocks in flight */
  for (; j < j1; j += B) {
    uint32_t kk[B];
    spmv_row<T> m[B];
    double xc[B];   /* a component a lane */
#pragma unroll
    for (uint32_t i = 0; i < B; i++) kk[i] = col[min(j + i, j1 - 1u)];
#pragma unroll
    for (uint32_t i = 0; i < B; i++) m[i].load(a + 16 * (size_t)min(j + i, j1 - 1u) + 4 * c);
#pragma unroll
    for (uint32_t i = 0; i < B; i++) xc[i] = x[4 * (size_t)kk[i] + c];
#pragma unroll
    for (uint32_t i = 0; i < B; i++) {
      double w[4];
      m[i].get(w);
      double s = acc + w[0] * spmv_quad<0>(xc[i]);
      s = s + w[1] * spmv_quad<1>(xc[i]);
      s = s + w[2] * spmv_quad<2>(xc[i]);
      s = s + w[3] * spmv_quad<3>(xc[i]);
      acc = j + i < j1 ? s : acc;
    }
  }
  y[4 * (size_t)r + c] = acc;
}

/* y = A x with the Jacobian ComputeA assembled last (the copy the context
 * keeps for the operator: FP64, or FP32 with a single-precision
 * preconditioner); x, y device vectors of 4N doubles, 32-byte aligned, not
 * aliased */
void kf_launch_spmv(kf_ctx *c, const double *x, double *y)
{
  kf_check_aligned(x, "x");
  kf_check_aligned(y, "y");
  const uint32_t nb = kf_blocks_for(c->d.N, SPMV_WG / 4);
  const int s = kf_prof_begin(c, KP_SPMV);
  if (c->jop64)
    hipLaunchKernelGGL(k_bsr_spmv<double>, dim3(nb), dim3(SPMV_WG), 0, c->stream, c->d.N, c->d.rowptr, c->d.col,
                       c->jop64, x, y);
  else
    hipLaunchKernelGGL(k_bsr_spmv<float>, dim3(nb), dim3(SPMV_WG), 0, c->stream, c->d.N, c->d.rowptr, c->d.col,
                       c->jop32, x, y);
  KF_LAUNCH_CHECK();
  kf_prof_end(c, s);
}
