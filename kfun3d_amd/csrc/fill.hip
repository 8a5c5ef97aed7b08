/*
 * fill.hip -- analytic first-order Jacobian A = J1 + diag(cdt) + boundary
 * blocks (src/fill.c:115-917, matrix/matrix.cpp:137-207) into BSR 4x4.
 *
 * One thread per block row.  The reference scatters the two edge blocks
 * v0, v1 of every edge into (n0,n0) += v0, (n0,n1) += v1, (n1,n0) -= v0,
 * (n1,n1) -= v1 in edge order, then adds the slip-wall column and the
 * free-stream block.  Here row v walks its incidences in ascending edge id,
 * recomputes v0 and v1 of each edge (cheaper than an HBM round trip of
 * 256 bytes per edge), accumulates its diagonal block in the reference's
 * order and writes each off-diagonal block exactly once.  The FP64 blocks
 * are bit-identical to the reference's; T = float gives the FP32
 * preconditioner matrix (inputs rounded to float, arithmetic in float).
 */
#include "kf_dev.h"

#define FLOAT_095 ((double)0.95f)

template <typename T>
__device__ __forceinline__ void edge_blocks(T xn, T yn, T zn, T ln, T uL, T vL, T wL, T uR, T vR, T wR, T v0[16],
                                            T v1[16])
{
  const T B = T(15), h = T(0.5), one = T(1);
  T dot = xn, X1, Y1, Z1;
  if (fabs((double)dot) < FLOAT_095) { X1 = one - dot * xn; Y1 = -dot * yn; Z1 = -dot * zn; }
  else { dot = yn; X1 = -dot * xn; Y1 = one - dot * yn; Z1 = -dot * zn; }
  T size = X1 * X1; size += Y1 * Y1; size += Z1 * Z1; size = sqrt(size);
  X1 /= size; Y1 /= size; Z1 /= size;
  T X2 = yn * Z1; X2 -= zn * Y1;
  T Y2 = zn * X1; Y2 -= xn * Z1;
  T Z2 = xn * Y1; Z2 -= yn * X1;
  T ubarL = xn * uL; ubarL += yn * vL; ubarL += zn * wL;
  T ubarR = xn * uR; ubarR += yn * vR; ubarR += zn * wR;
  const T u = h * (uL + uR), v = h * (vL + vR), w = h * (wL + wR);
  T ubar = xn * u; ubar += yn * v; ubar += zn * w;
  const T c2 = ubar * ubar + B;
  const T c = sqrt(c2);
  const T eig1 = ln * fabs(ubar), eig2 = ln * fabs(ubar), eig3 = ln * fabs(ubar + c), eig4 = ln * fabs(ubar - c);
  T phi1 = xn * B; phi1 += u * ubar;
  T phi2 = yn * B; phi2 += v * ubar;
  T phi3 = zn * B; phi3 += w * ubar;
  T phi4 = Y2 * phi3; phi4 -= Z2 * phi2;
  T phi5 = Z2 * phi1; phi5 -= X2 * phi3;
  T phi6 = X2 * phi2; phi6 -= Y2 * phi1;
  T phi7 = Z1 * phi2; phi7 -= Y1 * phi3;
  T phi8 = X1 * phi3; phi8 -= Z1 * phi1;
  T phi9 = Y1 * phi1; phi9 -= X1 * phi2;
  const T c2inv = one / c2;
  T y11 = u * phi4; y11 += v * phi5; y11 += w * phi6; y11 = -c2inv * y11 / B;
  T y21 = u * phi7; y21 += v * phi8; y21 += w * phi9; y21 = -c2inv * y21 / B;
  T y31 = c2inv * (c - ubar); y31 = h * y31 / B;
  T y41 = c2inv * (c + ubar); y41 = -h * y41 / B;
  const T y12 = c2inv * phi4, y22 = c2inv * phi7, y32 = c2inv * h * xn, y42 = c2inv * h * xn;
  const T y13 = c2inv * phi5, y23 = c2inv * phi8, y33 = c2inv * h * yn, y43 = c2inv * h * yn;
  const T y14 = c2inv * phi6, y24 = c2inv * phi9, y34 = c2inv * h * zn, y44 = c2inv * h * zn;
  const T t13 = c * B;
  T t23 = u * (ubar + c); t23 += xn * B;
  T t33 = v * (ubar + c); t33 += yn * B;
  T t43 = w * (ubar + c); t43 += zn * B;
  const T t14 = -c * B;
  T t24 = u * (ubar - c); t24 += xn * B;
  T t34 = v * (ubar - c); t34 += yn * B;
  T t44 = w * (ubar - c); t44 += zn * B;
  T a11 = eig3 * t13 * y31; a11 += eig4 * t14 * y41;
  T a12 = eig3 * t13 * y32; a12 += eig4 * t14 * y42;
  T a13 = eig3 * t13 * y33; a13 += eig4 * t14 * y43;
  T a14 = eig3 * t13 * y34; a14 += eig4 * t14 * y44;
  T a21 = eig1 * X1 * y11; a21 += eig2 * X2 * y21; a21 += eig3 * t23 * y31; a21 += eig4 * t24 * y41;
  T a22 = eig1 * X1 * y12; a22 += eig2 * X2 * y22; a22 += eig3 * t23 * y32; a22 += eig4 * t24 * y42;
  T a23 = eig1 * X1 * y13; a23 += eig2 * X2 * y23; a23 += eig3 * t23 * y33; a23 += eig4 * t24 * y43;
  T a24 = eig1 * X1 * y14; a24 += eig2 * X2 * y24; a24 += eig3 * t23 * y34; a24 += eig4 * t24 * y44;
  T a31 = eig1 * Y1 * y11; a31 += eig2 * Y2 * y21; a31 += eig3 * t33 * y31; a31 += eig4 * t34 * y41;
  T a32 = eig1 * Y1 * y12; a32 += eig2 * Y2 * y22; a32 += eig3 * t33 * y32; a32 += eig4 * t34 * y42;
  T a33 = eig1 * Y1 * y13; a33 += eig2 * Y2 * y23; a33 += eig3 * t33 * y33; a33 += eig4 * t34 * y43;
  T a34 = eig1 * Y1 * y14; a34 += eig2 * Y2 * y24; a34 += eig3 * t33 * y34; a34 += eig4 * t34 * y44;
  T a41 = eig1 * Z1 * y11; a41 += eig2 * Z2 * y21; a41 += eig3 * t43 * y31; a41 += eig4 * t44 * y41;
  T a42 = eig1 * Z1 * y12; a42 += eig2 * Z2 * y22; a42 += eig3 * t43 * y32; a42 += eig4 * t44 * y42;
  T a43 = eig1 * Z1 * y13; a43 += eig2 * Z2 * y23; a43 += eig3 * t43 * y33; a43 += eig4 * t44 * y43;
  T a44 = eig1 * Z1 * y14; a44 += eig2 * Z2 * y24; a44 += eig3 * t43 * y34; a44 += eig4 * t44 * y44;
  const T lb = ln * B, lx = ln * xn, ly = ln * yn, lz = ln * zn;
  v0[0] = h * a11; v0[4] = h * (lx + a21); v0[8] = h * (ly + a31); v0[12] = h * (lz + a41);
  v0[1] = h * ((lb * xn) + a12); v0[5] = h * ((ln * (ubarL + xn * uL)) + a22);
  v0[9] = h * ((lx * vL) + a32); v0[13] = h * ((lx * wL) + a42);
  v0[2] = h * ((lb * yn) + a13); v0[6] = h * ((ly * uL) + a23);
  v0[10] = h * ((ln * (ubarL + yn * vL)) + a33); v0[14] = h * ((ly * wL) + a43);
  v0[3] = h * ((lb * zn) + a14); v0[7] = h * ((lz * uL) + a24);
  v0[11] = h * ((lz * vL) + a34); v0[15] = h * ((ln * (ubarL + zn * wL)) + a44);
  v1[0] = h * -a11; v1[4] = h * (lx - a21); v1[8] = h * (ly - a31); v1[12] = h * (lz - a41);
  v1[1] = h * ((lb * xn) - a12); v1[5] = h * ((ln * (ubarR + xn * uR)) - a22);
  v1[9] = h * ((lx * vR) - a32); v1[13] = h * ((lx * wR) - a42);
  v1[2] = h * ((lb * yn) - a13); v1[6] = h * ((ly * uR) - a23);
  v1[10] = h * ((ln * (ubarR + yn * vR)) - a33); v1[14] = h * ((ly * wR) - a43);
  v1[3] = h * ((lb * zn) - a14); v1[7] = h * ((lz * uR) - a24);
  v1[11] = h * ((lz * vR) - a34); v1[15] = h * ((ln * (ubarR + zn * wR)) - a44);
}

/* free-stream characteristic block: src/fill.c:528-873 */
template <typename T>
__device__ __forceinline__ void freestream_block(T xn, T yn, T zn, T U, T V, T pi, T ui, T vi, T wi, T v[16])
{
  const T B = T(15), h = T(0.5), one = T(1), zero = T(0), W = T(0), P = T(1);
  const T ln = sqrt(xn * xn + yn * yn + zn * zn);
  xn /= ln; yn /= ln; zn /= ln;
  T dot = xn, X1, Y1, Z1;
  if (fabs((double)dot) < FLOAT_095) { X1 = one - dot * xn; Y1 = -dot * yn; Z1 = -dot * zn; }
  else { dot = yn; X1 = -dot * xn; Y1 = one - dot * yn; Z1 = -dot * zn; }
  const T size = sqrt(X1 * X1 + Y1 * Y1 + Z1 * Z1);
  X1 /= size; Y1 /= size; Z1 /= size;
  const T X2 = yn * Z1 - zn * Y1, Y2 = zn * X1 - xn * Z1, Z2 = xn * Y1 - yn * X1;
  T ubar0 = xn * U; ubar0 += yn * V; ubar0 += zn * W;
  const T c20 = ubar0 * ubar0 + B;
  const T c0 = sqrt(c20);
  T phi1 = xn * B; phi1 += U * ubar0;
  T phi2 = yn * B; phi2 += V * ubar0;
  T phi3 = zn * B; phi3 += W * ubar0;
  T phi4 = Y2 * phi3; phi4 -= Z2 * phi2;
  T phi5 = Z2 * phi1; phi5 -= X2 * phi3;
  T phi6 = X2 * phi2; phi6 -= Y2 * phi1;
  T phi7 = Z1 * phi2; phi7 -= Y1 * phi3;
  T phi8 = X1 * phi3; phi8 -= Z1 * phi1;
  T phi9 = Y1 * phi1; phi9 -= X1 * phi2;
  const T t13 = c0 * B;
  T t23 = U * (ubar0 + c0); t23 += xn * B;
  T t33 = V * (ubar0 + c0); t33 += yn * B;
  T t43 = W * (ubar0 + c0); t43 += zn * B;
  const T t14 = -c0 * B;
  T t24 = U * (ubar0 - c0); t24 += xn * B;
  T t34 = V * (ubar0 - c0); t34 += yn * B;
  T t44 = W * (ubar0 - c0); t44 += zn * B;
  T ti11 = U * phi4; ti11 += V * phi5; ti11 += W * phi6; ti11 = -ti11 / B / c20;
  T ti21 = U * phi7; ti21 += V * phi8; ti21 += W * phi9; ti21 = -ti21 / B / c20;
  const T ti31 = (c0 - ubar0) / (T(2) * B * c20);
  const T ti41 = -(c0 + ubar0) / (T(2) * B * c20);
  const T ti12 = phi4 / c20, ti22 = phi7 / c20, ti32 = h * xn / c20, ti42 = h * xn / c20;
  const T ti13 = phi5 / c20, ti23 = phi8 / c20, ti33 = h * yn / c20, ti43 = h * yn / c20;
  const T ti14 = phi6 / c20, ti24 = phi9 / c20, ti34 = h * zn / c20, ti44 = h * zn / c20;
  T un = xn * ui; un += yn * vi; un += zn * wi;
  T pr, prp, ur, uru, vr, vrv, wr, wrw;
  if (un > zero) { pr = pi; prp = one; ur = ui; uru = one; vr = vi; vrv = one; wr = wi; wrw = one; }
  else { pr = P; prp = zero; ur = U; uru = zero; vr = V; vrv = zero; wr = W; wrw = zero; }
  T rhs1 = ti11 * pr; rhs1 += ti12 * ur; rhs1 += ti13 * vr; rhs1 += ti14 * wr;
  const T rhs1p = ti11 * prp, rhs1u = ti12 * uru, rhs1v = ti13 * vrv, rhs1w = ti14 * wrw;
  T rhs2 = ti21 * pr; rhs2 += ti22 * ur; rhs2 += ti23 * vr; rhs2 += ti24 * wr;
  const T rhs2p = ti21 * prp, rhs2u = ti22 * uru, rhs2v = ti23 * vrv, rhs2w = ti24 * wrw;
  T rhs3 = ti31 * pi; rhs3 += ti32 * ui; rhs3 += ti33 * vi; rhs3 += ti34 * wi;
  T rhs4 = ti41 * P; rhs4 += ti42 * U; rhs4 += ti43 * V; rhs4 += ti44 * W;
  const T pbp = t13 * ti31, pbu = t13 * ti32, pbv = t13 * ti33, pbw = t13 * ti34;
  T ub = X1 * rhs1; ub += X2 * rhs2; ub += t23 * rhs3; ub += t24 * rhs4;
  T ubp = X1 * rhs1p; ubp += X2 * rhs2p; ubp += t23 * ti31;
  T ubu = X1 * rhs1u; ubu += X2 * rhs2u; ubu += t23 * ti32;
  T ubv = X1 * rhs1v; ubv += X2 * rhs2v; ubv += t23 * ti33;
  T ubw = X1 * rhs1w; ubw += X2 * rhs2w; ubw += t23 * ti34;
  T vb = Y1 * rhs1; vb += Y2 * rhs2; vb += t33 * rhs3; vb += t34 * rhs4;
  T vbp = Y1 * rhs1p; vbp += Y2 * rhs2p; vbp += t33 * ti31;
  T vbu = Y1 * rhs1u; vbu += Y2 * rhs2u; vbu += t33 * ti32;
  T vbv = Y1 * rhs1v; vbv += Y2 * rhs2v; vbv += t33 * ti33;
  T vbw = Y1 * rhs1w; vbw += Y2 * rhs2w; vbw += t33 * ti34;
  T wb = Z1 * rhs1; wb += Z2 * rhs2; wb += t43 * rhs3; wb += t44 * rhs4;
  T wbp = Z1 * rhs1p; wbp += Z2 * rhs2p; wbp += t43 * ti31;
  T wbu = Z1 * rhs1u; wbu += Z2 * rhs2u; wbu += t43 * ti32;
  T wbv = Z1 * rhs1v; wbv += Z2 * rhs2v; wbv += t43 * ti33;
  T wbw = Z1 * rhs1w; wbw += Z2 * rhs2w; wbw += t43 * ti34;
  T unb = xn * ub; unb += yn * vb; unb += zn * wb;
  T unbp = xn * ubp; unbp += yn * vbp; unbp += zn * wbp;
  T unbu = xn * ubu; unbu += yn * vbu; unbu += zn * wbu;
  T unbv = xn * ubv; unbv += yn * vbv; unbv += zn * wbv;
  T unbw = xn * ubw; unbw += yn * vbw; unbw += zn * wbw;
  v[0] = ln * B * unbp;
  v[4] = ln * (ub * unbp + unb * ubp + xn * pbp);
  v[8] = ln * (vb * unbp + unb * vbp + yn * pbp);
  v[12] = ln * (wb * unbp + unb * wbp + zn * pbp);
  v[1] = ln * B * unbu;
  v[5] = ln * (ub * unbu + unb * ubu + xn * pbu);
  v[9] = ln * (vb * unbu + unb * vbu + yn * pbu);
  v[13] = ln * (wb * unbu + unb * wbu + zn * pbu);
  v[2] = ln * B * unbv;
  v[6] = ln * (ub * unbv + unb * ubv + xn * pbv);
  v[10] = ln * (vb * unbv + unb * vbv + yn * pbv);
  v[14] = ln * (wb * unbv + unb * wbv + zn * pbv);
  v[3] = ln * B * unbw;
  v[7] = ln * (ub * unbw + unb * ubw + xn * pbw);
  v[11] = ln * (vb * unbw + unb * vbw + yn * pbw);
  v[15] = ln * (wb * unbw + unb * wbw + zn * pbw);
}

/* Blocks are stored by the whole wavefront through its own LDS: each lane
 * puts its block into its row (padded by 16 bytes, which say what to store
 * and keep the rows apart in the banks), then 8 lanes together store one
 * 128-byte line.  A lane storing its whole block by itself made 64 write
 * requests of 16 bytes an instruction, and those, 29 million at 496K
 * vertices, were what the kernel waited for.  An FP32 block is half a line,
 * and lines written in halves go to memory at 2.5 TB/s: a block waits in its
 * row for the other half of its line, which is the next incidence's wherever
 * edges ascend with their ends. */
template <typename T>
struct fill_rows {
  static constexpr int STRIDE = 9;   /* 16-byte pieces of a row */
  float4 w[64 * STRIDE];
};

#define FILL_NONE 0xffffffffu

/* the rows' lines: line in units of 128 bytes, FILL_NONE for no line, and the
 * halves that are there */
template <typename T>
__device__ __forceinline__ void store_lines(fill_rows<T> &rows, T *__restrict__ a, T *__restrict__ keep, uint32_t line,
                                            uint32_t halves)
{
  constexpr int STRIDE = fill_rows<T>::STRIDE;
  const uint32_t lane = threadIdx.x & 63u, piece = lane & 7u;
  float4 *o = rows.w + lane * STRIDE + 8;
  o->x = __uint_as_float(line);
  o->y = __uint_as_float(halves);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   /* the wavefront's own rows: in order, no barrier */
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 *in = rows.w + (i * 8 + lane / 8) * STRIDE;
    const float4 val = in[piece];
    const float2 w = *reinterpret_cast<const float2 *>(in + 8);
    const uint32_t n = __float_as_uint(w.x);
    if (n != FILL_NONE && (__float_as_uint(w.y) >> (piece >> 2) & 1u)) {
      reinterpret_cast<float4 *>(a + (128 / sizeof(T)) * (size_t)n)[piece] = val;
      if (keep) reinterpret_cast<float4 *>(keep + (128 / sizeof(T)) * (size_t)n)[piece] = val;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

/* FP64: a block is a line */
__device__ __forceinline__ void store_blocks(fill_rows<double> &rows, double *__restrict__ a,
                                             double *__restrict__ keep, uint32_t blk, const double v[16], uint32_t &,
                                             uint32_t &)
{
  double2 *o = reinterpret_cast<double2 *>(rows.w + (threadIdx.x & 63u) * fill_rows<double>::STRIDE);
#pragma unroll
  for (int k = 0; k < 8; k++) o[k] = make_double2(v[2 * k], v[2 * k + 1]);
  store_lines<double>(rows, a, keep, blk, 3u);
}

/* FP32: line, halves: what waits in the lane's row */
__device__ __forceinline__ void store_blocks(fill_rows<float> &rows, float *__restrict__ a, float *__restrict__ keep,
                                             uint32_t blk, const float v[16], uint32_t &line, uint32_t &halves)
{
  const bool other = blk != FILL_NONE && line != blk >> 1;   /* also when nothing waits */
  store_lines<float>(rows, a, keep, other ? line : FILL_NONE, halves);
  if (other) { line = blk >> 1; halves = 0u; }
  if (blk != FILL_NONE) {
    float4 *o = rows.w + (threadIdx.x & 63u) * fill_rows<float>::STRIDE + 4 * (blk & 1u);
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    halves |= 1u << (blk & 1u);
  }
}

/* Bound by memory: the records of the incidences once (40 bytes each, dense)
 * and the blocks once, at the rate of a copy.  173x61x47 (496K vertices), FP32
 * with the kept copy: 0.303 ms, 4.4 TB/s (0.379 ms and a copy of 0.126 ms with
 * lanes storing their own blocks and gathered edge records; 0.374 ms with
 * lines in halves); 144x48x48 FP64: 0.327 -> 0.190 ms.  More or fewer
 * wavefronts (2 to 4 a SIMD) make no difference.
 * keep: a second copy of the matrix, or NULL; a copy afterwards reads back
 * what was just written */
template <typename T>
__global__ __launch_bounds__(128) void k_fill(kf_dv d, const double *__restrict__ q, const double *__restrict__ cdt,
                                              T *__restrict__ a, T *__restrict__ keep)
{
  __shared__ fill_rows<T> srows[2];
  fill_rows<T> &rows = srows[threadIdx.x >> 6];
  const uint32_t t = kf_xcd_block() * 128u + threadIdx.x;
  const uint32_t slice = __builtin_amdgcn_readfirstlane(t >> 6);
  if (slice >= d.nslice) return;
  const uint32_t base = d.sell_ptr[slice], width = d.sell_ptr[slice + 1] - base;
  /* lanes behind the last row go along with no incidence */
  const uint32_t r = min(t, d.N - 1), deg = t < d.N ? d.deg[r] : 0u;
  const T zero = T(0), mone = T(-1);
  T dg[16];
#pragma unroll
  for (int k = 0; k < 16; k++) dg[k] = zero;
  const T cd = (T)cdt[r];
  dg[0] += cd; dg[5] += cd; dg[10] += cd; dg[15] += cd;
  const double *qr = q + 4 * (size_t)r;
  const T ur = (T)qr[1], vr = (T)qr[2], wr = (T)qr[3];
  /* The next incidence is loaded before this one is stored: loads behind
   * stores come back behind them, since one counter waits for both. */
  size_t idx = (size_t)base * 64u + (t & 63u);
  uint32_t nbs = 0, nbs1 = 0, blk1 = 0;   /* this incidence's, the next one's */
  uint32_t line = FILL_NONE, halves = 0;
  double qn[3];
  kf_egeo eg;
  if (width) {
    nbs = d.sell_nbs[idx];
    nbs1 = d.sell_nbs[width > 1 ? idx + 64 : idx];
    blk1 = d.sell_blk[idx];
    eg = kf_edge_geo(d.sell_geo, idx);
    const double *p = q + 4 * (size_t)(nbs & 0x7fffffffu);
    qn[0] = p[1]; qn[1] = p[2]; qn[2] = p[3];
  }
  for (uint32_t k = 0; k < width; k++, idx += 64) {
    T off[16];
    const T un = (T)qn[0], vn = (T)qn[1], wn = (T)qn[2];
    const T xn = (T)eg.xn, yn = (T)eg.yn, zn = (T)eg.zn, ln = (T)eg.ln;
    const bool side1 = nbs >> 31;
    const uint32_t blk = k < deg ? blk1 : FILL_NONE;
    if (k + 1 < width) {
      const double *p = q + 4 * (size_t)(nbs1 & 0x7fffffffu);
      qn[0] = p[1]; qn[1] = p[2]; qn[2] = p[3];
      eg = kf_edge_geo(d.sell_geo, idx + 64);
      nbs = nbs1;
      blk1 = d.sell_blk[idx + 64];
      nbs1 = d.sell_nbs[k + 2 < width ? idx + 128 : idx + 64];
    }
    if (k < deg) {
      /* r is n1: (n1,n0) -= v0, (n1,n1) -= v1; r is n0: (n0,n0) += v0, (n0,n1) += v1 */
      T v0[16], v1[16];
      edge_blocks<T>(xn, yn, zn, ln, side1 ? un : ur, side1 ? vn : vr, side1 ? wn : wr, side1 ? ur : un,
                     side1 ? vr : vn, side1 ? wr : wn, v0, v1);
#pragma unroll
      for (int j = 0; j < 16; j++) {
        off[j] = zero + (side1 ? mone * v0[j] : v1[j]);
        dg[j] += side1 ? mone * v1[j] : v0[j];
      }
    }
    store_blocks(rows, a, keep, blk, off, line, halves);
  }
  if (t < d.N) {
    for (uint32_t s = d.snptr[r]; s < d.snptr[r + 1]; s++) {   /* matrix/matrix.cpp:282-296 */
      const uint32_t i = d.snent[s];
      dg[4] += (T)d.snx[i]; dg[8] += (T)d.sny[i]; dg[12] += (T)d.snz[i];
    }
    for (uint32_t s = d.fnptr[r]; s < d.fnptr[r + 1]; s++) {
      const uint32_t i = d.fnent[s];
      T v[16];
      freestream_block<T>((T)d.fnx[i], (T)d.fny[i], (T)d.fnz[i], (T)d.U, (T)d.V, (T)qr[0], ur, vr, wr, v);
#pragma unroll
      for (int j = 0; j < 16; j++) dg[j] += v[j];
    }
  }
  store_blocks(rows, a, keep, t < d.N ? d.diag[r] : FILL_NONE, dg, line, halves);
  if (sizeof(T) == 4) store_lines<T>(rows, a, keep, line, halves);
}

static void ensure_f32(kf_ctx *c)
{
  if (!c->a32) KF_CHECK(hipMalloc((void **)&c->a32, 16 * c->nnzb * sizeof(float)));
}

/* the copy of the assembled Jacobian that the BSR operator reads (the ILU
 * factors the fill's array in place): room for it in the fill's precision */
static void ensure_kept(kf_ctx *c, bool f64)
{
  const size_t n = 16 * c->nnzb;
  if (f64 ? c->jop32 != NULL : c->jop64 != NULL) {
    /* the precision changed: drop the other copy (its last reader is done
     * once the stream is) */
    KF_CHECK(hipStreamSynchronize(c->stream));
    KF_CHECK(hipFree(f64 ? (void *)c->jop32 : (void *)c->jop64));
    c->jop32 = NULL;
    c->jop64 = NULL;
  }
  if (f64 && !c->jop64) KF_CHECK(hipMalloc((void **)&c->jop64, n * sizeof(double)));
  if (!f64 && !c->jop32) KF_CHECK(hipMalloc((void **)&c->jop32, n * sizeof(float)));
}

void kf_launch_fill(kf_ctx *c)
{
  const uint32_t nb = kf_blocks_for(c->d.N, 128);
  const bool f64 = c->opt.prec == KF_PREC_FP64, keep = c->opt.bsr_operator;
  if (keep) ensure_kept(c, f64);
  const int s = kf_prof_begin(c, KP_FILL);
  if (f64) {
    hipLaunchKernelGGL(k_fill<double>, dim3(nb), dim3(128), 0, c->stream, c->d, c->q, c->cdt, c->a64,
                       keep ? c->jop64 : (double *)NULL);
  } else {
    ensure_f32(c);
    hipLaunchKernelGGL(k_fill<float>, dim3(nb), dim3(128), 0, c->stream, c->d, c->q, c->cdt, c->a32,
                       keep ? c->jop32 : (float *)NULL);
  }
  KF_LAUNCH_CHECK();
  kf_prof_end(c, s);
}
