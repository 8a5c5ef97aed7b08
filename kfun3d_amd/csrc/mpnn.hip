/*
 * mpnn.hip -- the learned preconditioner's edge message-passing network on
 * gfx950: forward, backward (parameter gradients) and Adam.
 *
 * The network turns the ILU(0) factor's diagonal blocks and the mesh
 * geometry into a sparse linear correction operator G; the preconditioner
 * is M v = z + G z with z = ILU(0)^-1 v, linear in v.  Context (per vertex
 * v; u over v's neighbours in ascending edge order, e_vu the edge's unit
 * normal times its area, + when v is the edge's first vertex):
 *   x_v   = D_v / sd                                  16 features
 *   h0_v  = relu(W0 x_v + b0)                          32
 *   round l = 0..2:
 *     m_v = mean_u relu(A_l h_v + B_l h_u + C_l e_vu + c_l)
 *     h_v = h_v + relu(U_l h_v + V_l m_v + u_l)
 * Operator heads (16 values = one 4 x 4 block, row-major):
 *   [S_v; P_v] = WSA h_v + bSA,   Q_v = Wb h_v,   T_vu = P_v + Q_u + We e_vu
 * Correction:
 *   delta_v = S_v z_v + (1 / deg v) sum_u T_vu z_u
 * D_v is the diagonal block as stored (the inverse of U(v,v)) and sd the
 * RMS of all D blocks.  The context runs once per factorisation
 * (kf_mpnn_prepare); applying G is one gather over the incidence lists.
 *
 * Dense layers -- forward (W0, A_l, B_l, [U_l V_l], WSA, Wb), the data
 * gradients of backward and every weight gradient -- run on the matrix
 * cores: v_mfma_f32_32x32x8_bf16 with both operands rounded to bfloat16 and
 * FP32 accumulation.  Messages, the operator application and its backward
 * and the loss are FP32 vector code; every sum has a fixed order (per-vertex
 * gathers over the sliced-ELL incidence in ascending edge order, fixed
 * vertex partitions, fixed-tree and index-order reductions), so the network,
 * its gradient and its training are deterministic.
 *
 * Parameters are one FP32 vector in the order W0 b0 {A B C c U V u}x3
 * WSA bSA Wb We; it is the master copy Adam updates, and the bf16 copies
 * the matrix cores read are repacked after every update.
 */
#include <math.h>
#include <string.h>

#include "sync.h"

#define MP_H 32
#define MP_NIN 16 /* inputs: one diagonal block (a multiple of the MFMA k-step) */
#define MP_NR 3

/* offsets into the parameter vector */
#define MP_W0 0
#define MP_B0 (MP_W0 + MP_H * MP_NIN)
#define MP_R0 (MP_B0 + MP_H)
#define MP_RSZ (4 * MP_H * MP_H + MP_H * 3 + 2 * MP_H)
#define MP_A(l) (MP_R0 + (l) * MP_RSZ)
#define MP_B(l) (MP_A(l) + MP_H * MP_H)
#define MP_C(l) (MP_B(l) + MP_H * MP_H)
#define MP_CB(l) (MP_C(l) + MP_H * 3)
#define MP_U(l) (MP_CB(l) + MP_H)
#define MP_V(l) (MP_U(l) + MP_H * MP_H)
#define MP_UB(l) (MP_V(l) + MP_H * MP_H)
#define MP_WSA (MP_R0 + MP_NR * MP_RSZ) /* 32 x 32: S (rows 0-15), P (16-31) */
#define MP_BSA (MP_WSA + 32 * MP_H)
#define MP_WB (MP_BSA + 32)             /* 16 x 32: Q */
#define MP_WE (MP_WB + 16 * MP_H)       /* 16 x 3 */
#define MP_NPARAM (MP_WE + 16 * 3)
#define MP_HEADS (MP_NPARAM - MP_WSA)

static_assert(MP_NPARAM == 14928, "parameter layout of the network");

/* bf16 copies for the matrix cores, row-major [out][k].  Forward: W0
 * (32 x 16), per round A, B (32 x 32) and [U V] (32 x 64), then WSA and Wb
 * padded to 32 rows.  Backward (transposed): per round U^T, V^T (32 x 32)
 * and [A^T B^T] (32 x 64), then [WSA^T Wb^T] (32 x 64, Wb^T padded). */
#define MPB_W0 0
#define MPB_A(l) (MP_H * MP_NIN + (l) * 4 * MP_H * MP_H)
#define MPB_B(l) (MPB_A(l) + MP_H * MP_H)
#define MPB_UV(l) (MPB_B(l) + MP_H * MP_H)
#define MPB_WSA (MP_H * MP_NIN + MP_NR * 4 * MP_H * MP_H)
#define MPB_WB (MPB_WSA + MP_H * MP_H)
#define MPB_FWD (MPB_WB + MP_H * MP_H)
#define MPB_UT(l) (MPB_FWD + (l) * 4 * MP_H * MP_H)
#define MPB_VT(l) (MPB_UT(l) + MP_H * MP_H)
#define MPB_ABT(l) (MPB_VT(l) + MP_H * MP_H)
#define MPB_HT (MPB_FWD + MP_NR * 4 * MP_H * MP_H)
#define MPB_SIZE (MPB_HT + 2 * MP_H * MP_H)

#define MP_PARTS 1024 /* vertex partitions of the gradient reductions */
#define MP_RB 256

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 hwbf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float x)
{
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u); /* round to nearest, ties to even */
  return (unsigned short)(u >> 16);
}

/* ---- the context network's dense layers, 32 vertices per wavefront ------------
 *
 * Layers that follow one another on the same vertices run in one kernel on
 * registers.  The product is formed transposed, D = W X^T, so that lane l
 * holds vertex row0 + l % 32 and D's register 4 q + j holds output channel
 * 8 q + 4 (l / 32) + j -- exactly the B operand of the next layer's k-step q,
 * with no exchange between lanes; memory sees 16-byte loads and stores.
 * Operand layout of v_mfma_f32_32x32x8_bf16 (lane l, element j < 4):
 *   A: W[l % 32][8 s + 4 (l / 32) + j]
 *   B: X[row0 + l % 32][8 s + 4 (l / 32) + j]
 * The k-steps run in ascending s from a zero accumulator.  Bound by
 * the activations' bytes (backward reads them all): the first kernel moves
 * 640 bytes a vertex, a round 768.  331,776 vertices: 46 us and 68 us (3.8
 * TB/s) against 115 us (features and three layers) and 185 us (three layers)
 * with a kernel per layer; 112,035: 17 and 22 us against 56 and 73 us. */
__device__ __forceinline__ bf16x4 mp_bf4(const float *x)
{
  const f32x4 f = {x[0], x[1], x[2], x[3]};
  union { hwbf4 h; bf16x4 s; } u;
  u.h = __builtin_convertvector(f, hwbf4);   /* v_cvt_pk_bf16_f32: to nearest, ties to even */
  return u.s;
}

/* acc += W[.][k0 ...] x for S k-steps; x: the lane's 4 S channels, W row-major
 * with row stride K */
template <int S, int K>
__device__ __forceinline__ f32x16 mp_mm(const unsigned short *__restrict__ W, int k0, const float *x, f32x16 acc)
{
  const uint32_t li = threadIdx.x & 31u, h4 = (threadIdx.x & 32u) >> 3;
#pragma unroll
  for (int s = 0; s < S; s++) {
    const bf16x4 a = *reinterpret_cast<const bf16x4 *>(W + li * K + k0 + 8 * s + h4);
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, mp_bf4(x + 4 * s), acc, 0, 0, 0);
  }
  return acc;
}

__device__ __forceinline__ f32x16 mp_zero()
{
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = 0.0f;
  return z;
}

/* the lane's 16 channels of row n of a [N][32] array, and back */
__device__ __forceinline__ void mp_row_ld(const float *__restrict__ X, uint32_t n, float x[16])
{
  const float4 *p = reinterpret_cast<const float4 *>(X + (size_t)n * MP_H + ((threadIdx.x & 32u) >> 3));
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float4 t = p[2 * q];
    x[4 * q] = t.x; x[4 * q + 1] = t.y; x[4 * q + 2] = t.z; x[4 * q + 3] = t.w;
  }
}

__device__ __forceinline__ void mp_row_st(float *__restrict__ X, uint32_t n, const float x[16])
{
  float4 *p = reinterpret_cast<float4 *>(X + (size_t)n * MP_H + ((threadIdx.x & 32u) >> 3));
#pragma unroll
  for (int q = 0; q < 4; q++) p[2 * q] = make_float4(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
}

/* acc + b per channel (b NULL: + 0) */
__device__ __forceinline__ void mp_bias(const f32x16 &acc, const float *__restrict__ b, float z[16])
{
  const float4 *p = reinterpret_cast<const float4 *>(b + ((threadIdx.x & 32u) >> 3));
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float4 t = b ? p[2 * q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    z[4 * q] = acc[4 * q] + t.x; z[4 * q + 1] = acc[4 * q + 1] + t.y;
    z[4 * q + 2] = acc[4 * q + 2] + t.z; z[4 * q + 3] = acc[4 * q + 3] + t.w;
  }
}

#define MP_TW (MP_RB / 64)   /* tiles of 32 vertices per workgroup, one per wavefront */

/* x = D / sd, z0 = W0 x + b0, h = relu(z0), P = A h, Q = B h */
__global__ __launch_bounds__(MP_RB) void k_mp_in(uint32_t N, const float *__restrict__ D,
                                                 const float *__restrict__ isd_p, const unsigned short *__restrict__ wb,
                                                 const float *__restrict__ theta, float *__restrict__ X,
                                                 float *__restrict__ Z0, float *__restrict__ H, float *__restrict__ P,
                                                 float *__restrict__ Q)
{
  const uint32_t v = (kf_xcd_block() * MP_TW + (threadIdx.x >> 6)) * 32u + (threadIdx.x & 31u);
  const uint32_t n = min(v, N - 1), h4 = (threadIdx.x & 32u) >> 3;
  const bool on = v < N;
  const float isd = *isd_p;
  float x[8], z[16], y[16];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const float4 t = *reinterpret_cast<const float4 *>(D + (size_t)n * MP_NIN + 8 * s + h4);
    x[4 * s] = t.x * isd; x[4 * s + 1] = t.y * isd; x[4 * s + 2] = t.z * isd; x[4 * s + 3] = t.w * isd;
    if (on)
      *reinterpret_cast<float4 *>(X + (size_t)n * MP_NIN + 8 * s + h4) =
          make_float4(x[4 * s], x[4 * s + 1], x[4 * s + 2], x[4 * s + 3]);
  }
  mp_bias(mp_mm<2, MP_NIN>(wb + MPB_W0, 0, x, mp_zero()), theta + MP_B0, z);
#pragma unroll
  for (int r = 0; r < 16; r++) y[r] = fmaxf(z[r], 0.0f);
  if (on) { mp_row_st(Z0, n, z); mp_row_st(H, n, y); }
  mp_bias(mp_mm<4, MP_H>(wb + MPB_A(0), 0, y, mp_zero()), NULL, z);
  if (on) mp_row_st(P, n, z);
  mp_bias(mp_mm<4, MP_H>(wb + MPB_B(0), 0, y, mp_zero()), NULL, z);
  if (on) mp_row_st(Q, n, z);
}

/* zu = U h + V m + u, h' = h + relu(zu), then P = W1 h' + b1 and Q = W2 h':
 * the next round's A and B, or after the last round the heads WSA and Wb */
__global__ __launch_bounds__(MP_RB) void k_mp_update(uint32_t N, const float *__restrict__ H,
                                                     const float *__restrict__ M, const unsigned short *__restrict__ UV,
                                                     const float *__restrict__ ub, const unsigned short *__restrict__ W1,
                                                     const float *__restrict__ b1, const unsigned short *__restrict__ W2,
                                                     float *__restrict__ ZU, float *__restrict__ Hn,
                                                     float *__restrict__ P, float *__restrict__ Q)
{
  const uint32_t v = (kf_xcd_block() * MP_TW + (threadIdx.x >> 6)) * 32u + (threadIdx.x & 31u);
  const uint32_t n = min(v, N - 1);
  const bool on = v < N;
  float h[16], m[16], z[16];
  mp_row_ld(H, n, h);
  mp_row_ld(M, n, m);
  f32x16 acc = mp_mm<4, 2 * MP_H>(UV, 0, h, mp_zero());
  mp_bias(mp_mm<4, 2 * MP_H>(UV, MP_H, m, acc), ub, z);
#pragma unroll
  for (int r = 0; r < 16; r++) h[r] = h[r] + fmaxf(z[r], 0.0f);
  if (on) { mp_row_st(ZU, n, z); mp_row_st(Hn, n, h); }
  mp_bias(mp_mm<4, MP_H>(W1, 0, h, mp_zero()), b1, z);
  if (on) mp_row_st(P, n, z);
  mp_bias(mp_mm<4, MP_H>(W2, 0, h, mp_zero()), NULL, z);
  if (on) mp_row_st(Q, n, z);
}

/* ---- weight gradients on the matrix cores --------------------------------------
 *
 * A weight gradient sum_n dY[n][o] X[n][k] is a product over vertices, whose
 * operands want a lane per channel; the dense layers hold a lane per vertex.
 * Each wavefront turns its 32 x 32 tiles in LDS: rows are channels, MP_TS
 * bfloat16 values apart (72 bytes: the rows of 32 lanes start in different
 * banks), and the sums stay in registers over all of the wavefront's tiles.
 * With one wavefront per 328 vertices reading both operands again from memory
 * for every gradient, a pair of them took 160 us a round on 331,776 vertices. */
#define MP_TS 36

template <int Q>
__device__ __forceinline__ void mp_tile_put(short *T, const float *x)
{
  const uint32_t li = threadIdx.x & 31u, h4 = (threadIdx.x & 32u) >> 3;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const bf16x4 b = mp_bf4(x + 4 * q);
#pragma unroll
    for (int j = 0; j < 4; j++) T[(8 * q + h4 + j) * MP_TS + li] = b[j];
  }
}

/* the operand of lane l for vertices 8 t + 4 (l / 32) + j: row `row`, or 0 */
__device__ __forceinline__ bf16x4 mp_tile_get(const short *T, uint32_t row, bool on, int t)
{
  const bf16x4 z = {0, 0, 0, 0};
  return on ? *reinterpret_cast<const bf16x4 *>(T + row * MP_TS + 8 * t + ((threadIdx.x & 32u) >> 3)) : z;
}

/* acc[o][k] += sum over the tile's vertices of A[o] B[k], o < OY, k < KX */
template <int OY, int KX>
__device__ __forceinline__ f32x16 mp_tile_mm(const short *A, const short *B, f32x16 acc)
{
  const uint32_t li = threadIdx.x & 31u;
#pragma unroll
  for (int t = 0; t < 4; t++)
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(mp_tile_get(A, OY < 32 ? min(li, OY - 1u) : li, OY == 32 || li < OY, t),
                                                   mp_tile_get(B, KX < 32 ? min(li, KX - 1u) : li, KX == 32 || li < KX, t),
                                                   acc, 0, 0, 0);
  return acc;
}

/* the workgroup's sums of a weight gradient (o < OY, k < KX) into
 * out[o KX + k], wavefronts in order; sh holds MP_TW x 1024 floats */
template <int OY, int KX>
__device__ __forceinline__ void mp_wsum(const f32x16 &acc, float *sh, float *__restrict__ out)
{
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) sh[(threadIdx.x >> 6) * 1024 + 64 * r + (threadIdx.x & 63u)] = acc[r];
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < 1024; e += MP_RB) {
    float t = 0.0f;
    for (int w = 0; w < MP_TW; w++) t += sh[1024 * w + e];
    const uint32_t r = e >> 6, o = 8 * (r >> 2) + ((e & 32u) >> 3) + (r & 3u), k = e & 31u;
    if (o < (uint32_t)OY && k < (uint32_t)KX) out[o * KX + k] = t;
  }
}

/* the workgroup's sums of the lanes' 16 channels over all vertices */
__device__ __forceinline__ void mp_bsum(const float b[16], float *sh, float *__restrict__ out)
{
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) {
    float x = b[r];
#pragma unroll
    for (int m = 1; m < 32; m <<= 1) x += __shfl_xor(x, m, 64);
    if ((threadIdx.x & 31u) == 0) sh[(threadIdx.x >> 6) * 32 + 8 * (r >> 2) + ((threadIdx.x & 32u) >> 3) + (r & 3)] = x;
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    float t = 0.0f;
    for (int w = 0; w < MP_TW; w++) t += sh[32 * w + threadIdx.x];
    out[threadIdx.x] = t;
  }
}

/* grad[i] = sum over partitions of part[p][i] (FP64): a workgroup takes 64
 * parameters, its 16 wavefronts every 16th partition each, then the
 * wavefronts in order (943 partitions: 30 us, against 396 us for one thread
 * per parameter) */
__global__ __launch_bounds__(1024) void k_mp_grad_reduce(const float *__restrict__ part, uint32_t nparts,
                                                         float *__restrict__ grad)
{
  __shared__ double sh[16][64];
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, i = blockIdx.x * 64u + lane;
  double acc = 0.0;
  if (i < MP_NPARAM)
    for (uint32_t p = w; p < nparts; p += 16) acc += (double)part[(size_t)p * MP_NPARAM + i];
  sh[w][lane] = acc;
  __syncthreads();
  if (w == 0 && i < MP_NPARAM) {
    for (int k = 1; k < 16; k++) acc += sh[k][lane];
    grad[i] = (float)acc;
  }
}

/* ---- reductions and features ---------------------------------------------------- */

__device__ __forceinline__ double mp_block_sum(double v, double *sh)
{
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
#pragma unroll
  for (int s = MP_RB / 2; s > 0; s >>= 1) {
    if (t < s) sh[t] = sh[t] + sh[t + s];
    __syncthreads();
  }
  return sh[0];
}

/* KF_NRED partial sums of squares (fixed grid and stride, fixed tree) */
template <typename T>
__global__ __launch_bounds__(MP_RB) void k_mp_sumsq(size_t n, const T *__restrict__ x, double *__restrict__ part)
{
  __shared__ double sh[MP_RB];
  double acc = 0.0;
  const size_t stride = (size_t)gridDim.x * MP_RB;
  for (size_t i = (size_t)blockIdx.x * MP_RB + threadIdx.x; i < n; i += stride) {
    const double v = (double)x[i];
    acc += v * v;
  }
  const double s = mp_block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

/* *out = 1 / RMS over `count` values from the KF_NRED partials (1 when zero or
 * not finite) */
__global__ __launch_bounds__(MP_RB) void k_mp_finish(const double *__restrict__ part, double count,
                                                     float *__restrict__ out)
{
  __shared__ double sh[MP_RB];
  double a = 0.0;
  for (int i = threadIdx.x; i < KF_NRED; i += MP_RB) a += part[i];
  a = mp_block_sum(a, sh);
  if (threadIdx.x != 0) return;
  double s = sqrt(a / count);
  if (!(s > 0.0) || !isfinite(s)) s = 1.0;
  *out = (float)(1.0 / s);
}

/* the ILU factor's diagonal blocks, as FP32 [N][16] */
template <typename TD>
__global__ __launch_bounds__(MP_RB) void k_mp_take_diag(uint32_t N, const uint32_t *__restrict__ diag,
                                                        const TD *__restrict__ a, float *__restrict__ D)
{
  const size_t k = (size_t)blockIdx.x * MP_RB + threadIdx.x;
  if (k >= 16 * (size_t)N) return;
  D[k] = (float)a[16 * (size_t)diag[k >> 4] + (k & 15)];
}

/* signed edge vector of every sliced-ELL slot: (nx, ny, nz) area, negated
 * where the vertex is the edge's second end; the fourth word holds the edge's
 * place in the neighbour's own list (an integer), where the backward pass
 * finds the message that went the other way */
__global__ __launch_bounds__(MP_RB) void k_mp_edge_vectors(kf_dv d, float4 *__restrict__ ev, float *__restrict__ ideg)
{
  const uint32_t v = blockIdx.x * MP_RB + threadIdx.x;
  if (v >= d.N) return;
  size_t idx = (size_t)d.sell_ptr[v >> 6] * 64u + (v & 63u);
  for (uint32_t k = 0; k < d.deg[v]; k++, idx += 64) {
    const uint32_t at = d.sell_pos[idx], u = d.sell_nbr[idx];
    const kf_egeo eg = kf_edge_geo(d.sell_geo, idx);
    const double ar = (at & 1u) ? -eg.ln : eg.ln;
    const size_t ui = (size_t)d.sell_ptr[u >> 6] * 64u + (u & 63u);
    uint32_t kr = 0;
    while (kr + 1 < d.deg[u] && d.sell_pos[ui + 64 * (size_t)kr] != (at ^ 1u)) kr++;   /* u holds the other side */
    ev[idx] = make_float4((float)(eg.xn * ar), (float)(eg.yn * ar), (float)(eg.zn * ar), __uint_as_float(kr));
  }
  ideg[v] = 1.0f / (float)max(d.deg[v], 1u);
}

/* ---- messages ------------------------------------------------------------------ */

/* Layout of both directions: 8 lanes per vertex, 4 channels per lane (one
 * 16-byte load of a 128-byte row each), 32 vertices per workgroup.  One load
 * instruction of a wavefront then reads 8 whole rows and the per-edge work
 * (neighbour index, edge vector, addresses) is shared by 4 channels.  On
 * 331,776 vertices a round takes 91 us forward and 137 us backward; with one
 * channel per lane and 2 vertices per wavefront the same sums took 258 and
 * 644 us (112,035 vertices forward: 27 against 73 us). */
#define MP_VW 32   /* vertices per workgroup of the message kernels */

__device__ __forceinline__ void mp_ld4(const float *__restrict__ p, float x[4])
{
  const float4 t = *reinterpret_cast<const float4 *>(p);
  x[0] = t.x; x[1] = t.y; x[2] = t.z; x[3] = t.w;
}

/* x where bit b of w is set, else +0, without a branch */
__device__ __forceinline__ float mp_keep(float x, uint32_t w, int b)
{
  return __uint_as_float(__float_as_uint(x) & (uint32_t)__builtin_amdgcn_sbfe((int)w, b, 1));
}

/* m_v = mean over v's incidences of relu(P_v + Q_u + C e_vu + c), and which
 * of them were positive: 4 bits per incidence and lane (bit j: channel 4 s +
 * j of lane s), 8 incidences per word, at pos[(v words + k / 8) 8 + s], for
 * the backward pass.  Four incidences' gathers are in flight together (slots
 * past the vertex's degree read its last one and count 0); the sums keep the
 * edge order.  Bound by the gathers' latency and L2 rate (14 rows of 128
 * bytes per vertex). */
__global__ __launch_bounds__(MP_RB) void k_mp_message(kf_dv d, const float4 *__restrict__ ev,
                                                      const float *__restrict__ P, const float *__restrict__ Q,
                                                      const float *__restrict__ theta, uint32_t offC, uint32_t offc,
                                                      float *__restrict__ M, uint32_t *__restrict__ pos,
                                                      uint32_t words)
{
  const uint32_t s = threadIdx.x & 7u, v = kf_xcd_block() * MP_VW + (threadIdx.x >> 3);
  if (v >= d.N) return;
  const uint32_t deg = d.deg[v];
  const size_t base = (size_t)d.sell_ptr[v >> 6] * 64u + (v & 63u);
  float cc[12], cb[4], pv[4], acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int i = 0; i < 3; i++) mp_ld4(theta + offC + 12 * s + 4 * i, cc + 4 * i);
  mp_ld4(theta + offc + 4 * s, cb);
  mp_ld4(P + (size_t)v * MP_H + 4 * s, pv);
  uint32_t word = 0;
  for (uint32_t k0 = 0; k0 < deg; k0 += 4) {
    uint32_t u[4];
    float4 e[4];
    float q[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const size_t idx = base + 64 * (size_t)min(k0 + i, deg - 1);
      u[i] = d.sell_nbr[idx];
      e[i] = ev[idx];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) mp_ld4(Q + (size_t)u[i] * MP_H + 4 * s, q[i]);
    const uint32_t sh = 4 * (k0 & 4u);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      /* relu(z), and 0 past the degree, without a branch: the median of z, 0 and the limit */
      const float lim = k0 + i < deg ? __builtin_inff() : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float z = pv[j] + q[i][j] + (cc[3 * j] * e[i].x + cc[3 * j + 1] * e[i].y + cc[3 * j + 2] * e[i].z) + cb[j];
        const float r = __builtin_amdgcn_fmed3f(z, 0.0f, lim);
        acc[j] += r;
        word |= (uint32_t)min(max(__float_as_int(r), 0), 1) << (sh + 4 * i + j);   /* r > 0 */
      }
      __builtin_amdgcn_sched_barrier(0);   /* one incidence's temporaries at a time: registers */
    }
    if ((k0 & 4u) || k0 + 4 >= deg) {
      pos[((size_t)v * words + (k0 >> 3)) * 8 + s] = word;
      word = 0;
    }
  }
  const float id = 1.0f / (float)max(deg, 1u);
  *reinterpret_cast<float4 *>(M + (size_t)v * MP_H + 4 * s) =
      make_float4(acc[0] * id, acc[1] * id, acc[2] * id, acc[3] * id);
}

/* Backward of the messages for partition p = blockIdx.x, MP_VW vertices at a
 * time.  With dm already divided by the degree:
 *   dP_v = sum_{(v,u)} dm_v [z_vu > 0]
 *   dQ_v = sum_{(v,u)} dm_u [z_uv > 0]     (the message u formed of v)
 * and the partition's sums of dm_v [z_vu > 0] e_vu and of dm_v [z_vu > 0]
 * (the gradients of C and c), reduced over the vertex groups in a fixed
 * order.  The signs come from the forward pass's bits (v's own words, and
 * the neighbour's word at the edge's place in its list), so a neighbour
 * costs its dm row and one word per lane instead of its P, Q and dm rows
 * and two recomputed messages. */
__global__ __launch_bounds__(MP_RB) void k_mp_message_bwd(kf_dv d, uint32_t chunk, const float4 *__restrict__ ev,
                                                          const uint32_t *__restrict__ pos, uint32_t words,
                                                          const float *__restrict__ dm, uint32_t offC, uint32_t offc,
                                                          float *__restrict__ dP, float *__restrict__ dQ,
                                                          float *__restrict__ part)
{
  __shared__ float sh[MP_RB / 64][8][16];
  const uint32_t s = threadIdx.x & 7u, grp = threadIdx.x >> 3;
  const uint32_t p = kf_xcd_block(), n0 = p * chunk, n1 = min(d.N, n0 + chunk);
  float g[4][3], gb[4];
#pragma unroll
  for (int j = 0; j < 4; j++) g[j][0] = g[j][1] = g[j][2] = gb[j] = 0.0f;
  for (uint32_t v = n0 + grp; v < n1; v += MP_VW) {
    const uint32_t deg = d.deg[v];
    const size_t base = (size_t)d.sell_ptr[v >> 6] * 64u + (v & 63u);
    float dmv[4], ap[4] = {0.0f, 0.0f, 0.0f, 0.0f}, aq[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    mp_ld4(dm + (size_t)v * MP_H + 4 * s, dmv);
    for (uint32_t k0 = 0; k0 < deg; k0 += 4) {
      uint32_t u[4], rb[4];
      float4 e[4];
      float dmu[4][4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const size_t idx = base + 64 * (size_t)min(k0 + i, deg - 1);
        u[i] = d.sell_nbr[idx];
        e[i] = ev[idx];
      }
      const uint32_t own = pos[((size_t)v * words + (k0 >> 3)) * 8 + s] >> (4 * (k0 & 4u));
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t kr = __float_as_uint(e[i].w);
        mp_ld4(dm + (size_t)u[i] * MP_H + 4 * s, dmu[i]);
        rb[i] = pos[((size_t)u[i] * words + (kr >> 3)) * 8 + s] >> (4 * (kr & 7u));
      }
#pragma unroll
      for (int i = 0; i < 4; i++) rb[i] = k0 + i < deg ? rb[i] : 0u;
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float gv = mp_keep(dmv[j], own, 4 * i + j);   /* bits past the degree are 0 */
          ap[j] += gv;
          g[j][0] += gv * e[i].x;
          g[j][1] += gv * e[i].y;
          g[j][2] += gv * e[i].z;
          gb[j] += gv;
          aq[j] += mp_keep(dmu[i][j], rb[i], j);
        }
      }
    }
    *reinterpret_cast<float4 *>(dP + (size_t)v * MP_H + 4 * s) = make_float4(ap[0], ap[1], ap[2], ap[3]);
    *reinterpret_cast<float4 *>(dQ + (size_t)v * MP_H + 4 * s) = make_float4(aq[0], aq[1], aq[2], aq[3]);
  }
  /* the wavefront's 8 vertex groups by lane exchange, then the wavefronts */
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float x = i < 3 ? g[j][i < 3 ? i : 0] : gb[j];
      x += __shfl_xor(x, 8, 64);
      x += __shfl_xor(x, 16, 64);
      x += __shfl_xor(x, 32, 64);
      if ((threadIdx.x & 63u) < 8) sh[threadIdx.x >> 6][s][4 * j + i] = x;
    }
  __syncthreads();
  if (threadIdx.x < MP_H * 4) {
    const uint32_t c = threadIdx.x >> 2, i = threadIdx.x & 3u;
    float t = 0.0f;
    for (int w = 0; w < MP_RB / 64; w++) t += sh[w][c >> 2][4 * (c & 3u) + i];
    float *pp = part + (size_t)p * MP_NPARAM;
    if (i < 3) pp[offC + 3 * c + i] = t;
    else pp[offc + c] = t;
  }
}

/* ---- the correction operator ------------------------------------------------------ */

__device__ __forceinline__ float4 ld4(const double *z, uint32_t v)
{
  return make_float4((float)z[4 * (size_t)v], (float)z[4 * (size_t)v + 1], (float)z[4 * (size_t)v + 2],
                     (float)z[4 * (size_t)v + 3]);
}

/* delta_v = S_v z_v + (1/deg v) [(P_v + b) zs_v + We : Ez_v + sum_u Q_u z_u]
 * with zs_v = sum_u z_u and Ez_v[j][k] = sum_u z_u[j] e_vu[k] (the edge
 * blocks T_vu = P_v + b + Q_u + We e_vu factored), one thread per vertex.
 * OP1 = [S | P + b] (N x 32), OPQ = [Q | 0] (N x 32).  Output: FP64 out
 * (stored, or added when add) or, when err is given, the FP32 error
 * err = z + delta - target (formed in FP64; target NULL: z + delta).  Two
 * neighbours' rows are in flight; the sums keep the edge order. */
__global__ __launch_bounds__(MP_RB) void k_mp_apply(kf_dv d, const float4 *__restrict__ ev,
                                                    const float *__restrict__ OP1, const float *__restrict__ OPQ,
                                                    const float *__restrict__ theta, const double *__restrict__ z,
                                                    double *__restrict__ out, int add,
                                                    const double *__restrict__ target, float *__restrict__ err)
{
  __shared__ float we[48];
  if (threadIdx.x < 48) we[threadIdx.x] = theta[MP_WE + threadIdx.x];
  __syncthreads();
  const uint32_t v = kf_xcd_block() * MP_RB + threadIdx.x;
  if (v >= d.N) return;
  const uint32_t deg = d.deg[v];
  size_t idx = (size_t)d.sell_ptr[v >> 6] * 64u + (v & 63u);
  float qz[4] = {0.0f, 0.0f, 0.0f, 0.0f}, zs[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ez[12];
#pragma unroll
  for (int i = 0; i < 12; i++) ez[i] = 0.0f;
  auto sum = [&](const float4 &e, const float4 &zu4, const float4 q[4]) {
    const float zu[4] = {zu4.x, zu4.y, zu4.z, zu4.w};
#pragma unroll
    for (int i = 0; i < 4; i++) qz[i] += q[i].x * zu[0] + q[i].y * zu[1] + q[i].z * zu[2] + q[i].w * zu[3];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      zs[j] += zu[j];
      ez[3 * j] += zu[j] * e.x;
      ez[3 * j + 1] += zu[j] * e.y;
      ez[3 * j + 2] += zu[j] * e.z;
    }
  };
  uint32_t k = 0;
  for (; k + 1 < deg; k += 2, idx += 128) {
    const uint32_t ua = d.sell_nbr[idx], ub = d.sell_nbr[idx + 64];
    const float4 ea = ev[idx], eb = ev[idx + 64];
    const float4 za = ld4(z, ua), zb = ld4(z, ub);
    const float4 *pa = (const float4 *)(OPQ + (size_t)ua * MP_H), *pb = (const float4 *)(OPQ + (size_t)ub * MP_H);
    const float4 qa[4] = {pa[0], pa[1], pa[2], pa[3]}, qb[4] = {pb[0], pb[1], pb[2], pb[3]};
    sum(ea, za, qa);
    sum(eb, zb, qb);
  }
  if (k < deg) {
    const uint32_t ua = d.sell_nbr[idx];
    const float4 ea = ev[idx], za = ld4(z, ua);
    const float4 *pa = (const float4 *)(OPQ + (size_t)ua * MP_H);
    const float4 qa[4] = {pa[0], pa[1], pa[2], pa[3]};
    sum(ea, za, qa);
  }
  const float4 zv4 = ld4(z, v);
  const float zv[4] = {zv4.x, zv4.y, zv4.z, zv4.w};
  const float *op = OP1 + (size_t)v * MP_H;
  const float idg = 1.0f / (float)max(deg, 1u);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float sv = 0.0f, t = qz[i];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      sv += op[4 * i + j] * zv[j];
      t += op[16 + 4 * i + j] * zs[j];
      t += we[3 * (4 * i + j)] * ez[3 * j] + we[3 * (4 * i + j) + 1] * ez[3 * j + 1] +
           we[3 * (4 * i + j) + 2] * ez[3 * j + 2];
    }
    const float dl = sv + t * idg;
    const size_t o = 4 * (size_t)v + i;
    if (err) err[o] = (float)(z[o] + (double)dl - (target ? target[o] : 0.0));
    else out[o] = add ? out[o] + (double)dl : (double)dl;
  }
}

/* ---- backward of the dense layers, per vertex partition -------------------------
 *
 * blockIdx.x is a partition of `chunk` vertices (a multiple of 32), its
 * wavefronts take tiles of 32 vertices in turn, and the layers of the context
 * network run backward on registers as in k_mp_update; the weight gradients
 * of the partition go to part[p].  Everything that follows on a vertex's own
 * values is one kernel; the messages' backward, which gathers, lies between.
 * Bound by the bytes: 1.1 KB a vertex and round, 91 us on 331,776 vertices
 * (4.1 TB/s), where a kernel per layer and gradient took 530 us.  The sums of
 * four gradients leave two wavefronts per SIMD (256 registers). */

/* dzu = dh where zu > 0; dhn = dh + dzu U, dm = (dzu V) / deg; tiles of dzu,
 * h and m for the gradients of U and V; bu += dzu */
__device__ __forceinline__ void mp_update_bwd(const float dh[16], uint32_t n, bool on, const float *__restrict__ ZU,
                                              const float *__restrict__ H, const float *__restrict__ M,
                                              const unsigned short *__restrict__ wut,
                                              const unsigned short *__restrict__ wvt, float idg,
                                              float *__restrict__ dhn, float *__restrict__ dm, short *T, float bu[16],
                                              f32x16 &gu, f32x16 &gv)
{
  float x[16], z[16];
  mp_row_ld(ZU, n, x);
#pragma unroll
  for (int r = 0; r < 16; r++) {
    x[r] = on && x[r] > 0.0f ? dh[r] : 0.0f;
    bu[r] += x[r];
  }
  mp_bias(mp_mm<4, MP_H>(wut, 0, x, mp_zero()), NULL, z);
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = dh[r] + z[r];
  if (on) mp_row_st(dhn, n, z);
  mp_bias(mp_mm<4, MP_H>(wvt, 0, x, mp_zero()), NULL, z);
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = z[r] * idg;
  if (on) mp_row_st(dm, n, z);
  wave_lds_sync();   /* the tiles' last readers are done */
  mp_tile_put<4>(T, x);
  mp_row_ld(H, n, z);
  mp_tile_put<4>(T + 32 * MP_TS, z);
  mp_row_ld(M, n, z);
  mp_tile_put<4>(T + 64 * MP_TS, z);
  wave_lds_sync();
  gu = mp_tile_mm<32, 32>(T, T + 32 * MP_TS, gu);
  gv = mp_tile_mm<32, 32>(T, T + 64 * MP_TS, gv);
}

#define MP_BWD_TILES (96 * MP_TS)   /* values: a wavefront's 3 tiles of 32 rows */
/* bytes: 6,912 a wavefront for its tiles, and after them 4,096 for its sums.
 * With no more than the tiles need the compiler's code for k_mp_head_bwd is
 * another, and slower (331,776 vertices: 147 against 135 us). */
#define MP_BWD_LDS (MP_TW * 8192)
static_assert(MP_BWD_LDS >= MP_TW * MP_BWD_TILES * 2 && MP_BWD_LDS >= MP_TW * 4096, "tiles and sums fit");

/* Backward of the correction given gv = dL/d delta (N x 4, FP32) and z:
 *   dOP1_v = [g_v z_v^T | (g_v / deg v) zs_v^T]       zs_v = sum_u z_u
 *   dOPQ_v = gbar_v z_v^T,  gbar_v = sum_u g_u / deg u
 *   gd_v   = g_v / deg v,  Ez_v[3 j + k] = sum_u z_u[j] e_vu[k]
 * (the gradient of We is sum_v gd_v Ez_v^T), the heads' weight gradients, dh
 * = dOP1 WSA + dOPQ Wb, and the last round's update backward (148 us on
 * 331,776 vertices; two gathers in flight took 197 us, separate kernels 470). */
__global__ __launch_bounds__(MP_RB, 2) void k_mp_head_bwd(kf_dv d, uint32_t chunk, const float4 *__restrict__ ev,
                                                       const float *__restrict__ ideg, const double *__restrict__ z,
                                                       const float *__restrict__ gv, const unsigned short *__restrict__ wb,
                                                       const float *__restrict__ Hl, const float *__restrict__ ZU,
                                                       const float *__restrict__ H, const float *__restrict__ M,
                                                       float *__restrict__ dhn, float *__restrict__ dm,
                                                       float *__restrict__ part)
{
  __shared__ __align__(16) unsigned char lds[MP_BWD_LDS];
  short *T = reinterpret_cast<short *>(lds) + (threadIdx.x >> 6) * MP_BWD_TILES;
  float *sh = reinterpret_cast<float *>(lds);
  const uint32_t li = threadIdx.x & 31u, hf = (threadIdx.x >> 5) & 1u;
  const uint32_t p = kf_xcd_block(), n0 = p * chunk, n1 = min(d.N, n0 + chunk);
  f32x16 gs = mp_zero(), gq = mp_zero(), ge = mp_zero(), gu = mp_zero(), gw = mp_zero();
  float bs[16], bu[16];
#pragma unroll
  for (int r = 0; r < 16; r++) bs[r] = bu[r] = 0.0f;
  for (uint32_t row = n0 + 32 * (threadIdx.x >> 6); row < n1; row += 32 * MP_TW) {
    const uint32_t v = min(row + li, n1 - 1);
    const bool on = row + li < n1;
    const uint32_t deg = d.deg[v];
    const size_t base = (size_t)d.sell_ptr[v >> 6] * 64u + (v & 63u);
    float zs[4] = {0.0f, 0.0f, 0.0f, 0.0f}, gb[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ez[12];
#pragma unroll
    for (int i = 0; i < 12; i++) ez[i] = 0.0f;
    /* four incidences' gathers in flight: at two wavefronts per SIMD their
     * latency is what this kernel waits for */
    for (uint32_t k0 = 0; k0 < deg; k0 += 4) {
      uint32_t u[4];
      float4 e[4], zu[4], gu4[4];
      float iu[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const size_t idx = base + 64 * (size_t)min(k0 + i, deg - 1);
        u[i] = d.sell_nbr[idx];
        e[i] = ev[idx];
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        zu[i] = ld4(z, u[i]);
        gu4[i] = *(const float4 *)(gv + 4 * (size_t)u[i]);
        iu[i] = ideg[u[i]];
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool in = k0 + i < deg;
        const float zz[4] = {in ? zu[i].x : 0.0f, in ? zu[i].y : 0.0f, in ? zu[i].z : 0.0f, in ? zu[i].w : 0.0f};
        gb[0] += (in ? gu4[i].x : 0.0f) * iu[i];
        gb[1] += (in ? gu4[i].y : 0.0f) * iu[i];
        gb[2] += (in ? gu4[i].z : 0.0f) * iu[i];
        gb[3] += (in ? gu4[i].w : 0.0f) * iu[i];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          zs[j] += zz[j];
          ez[3 * j] += zz[j] * e[i].x;
          ez[3 * j + 1] += zz[j] * e[i].y;
          ez[3 * j + 2] += zz[j] * e[i].z;
        }
      }
    }
    const float4 zv4 = ld4(z, v), g4 = *(const float4 *)(gv + 4 * (size_t)v);
    const float idg = ideg[v];
    const float zv[4] = {zv4.x, zv4.y, zv4.z, zv4.w}, g[4] = {g4.x, g4.y, g4.z, g4.w};
    float gi[4], x1[16], x2[8], x3[12];
#pragma unroll
    for (int i = 0; i < 4; i++) gi[i] = on ? g[i] * idg : 0.0f;
    /* the lane's channels 8 q + 4 (lane / 32) + j: row 2 q + lane / 32 of the
     * 4 x 4 blocks, column j */
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const float a = on ? (hf ? g[2 * q + 1] : g[2 * q]) : 0.0f, b = hf ? gi[2 * q + 1] : gi[2 * q];
      const float c = on ? (hf ? gb[2 * q + 1] : gb[2 * q]) : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        x1[4 * q + j] = a * zv[j];
        x1[8 + 4 * q + j] = b * zs[j];
        x2[4 * q + j] = c * zv[j];
      }
    }
#pragma unroll
    for (int r = 0; r < 16; r++) bs[r] += x1[r];
    float hl[16], dh[16];
    mp_row_ld(Hl, v, hl);
    f32x16 acc = mp_mm<4, 2 * MP_H>(wb + MPB_HT, 0, x1, mp_zero());
    acc = mp_mm<2, 2 * MP_H>(wb + MPB_HT, MP_H, x2, acc);   /* the padded half of Wb^T is 0 */
    mp_bias(acc, NULL, dh);
    wave_lds_sync();
    mp_tile_put<4>(T, x1);
    mp_tile_put<2>(T + 32 * MP_TS, x2);
    mp_tile_put<4>(T + 64 * MP_TS, hl);
    /* rows 48 .. 63: Ez (12) and gd (4), 8 per half */
#pragma unroll
    for (int i = 0; i < 12; i++) x3[i] = ez[i];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float y[4] = {hf ? x3[4 + j] : x3[j], hf ? x3[8 + j] : gi[j], 0.0f, 0.0f};
      const bf16x4 b = mp_bf4(y);
      T[(48 + (hf ? 4 : 0) + j) * MP_TS + li] = b[0];
      T[(48 + (hf ? 8 : 12) + j) * MP_TS + li] = b[1];
    }
    wave_lds_sync();
    gs = mp_tile_mm<32, 32>(T, T + 64 * MP_TS, gs);
    gq = mp_tile_mm<16, 32>(T + 32 * MP_TS, T + 64 * MP_TS, gq);
    ge = mp_tile_mm<4, 12>(T + 60 * MP_TS, T + 48 * MP_TS, ge);
    mp_update_bwd(dh, v, on, ZU, H, M, wb + MPB_UT(MP_NR - 1), wb + MPB_VT(MP_NR - 1), idg, dhn, dm, T, bu, gu, gw);
  }
  float *pp = part + (size_t)p * MP_NPARAM;
  mp_wsum<32, MP_H>(gs, sh, pp + MP_WSA);
  mp_bsum(bs, sh, pp + MP_BSA);
  mp_wsum<16, MP_H>(gq, sh, pp + MP_WB);
  mp_wsum<4, 12>(ge, sh, pp + MP_WE);
  mp_wsum<MP_H, MP_H>(gu, sh, pp + MP_U(MP_NR - 1));
  mp_wsum<MP_H, MP_H>(gw, sh, pp + MP_V(MP_NR - 1));
  mp_bsum(bu, sh, pp + MP_UB(MP_NR - 1));
}

/* After round l's messages: the gradients of A_l and B_l, dh = dhn + dP A +
 * dQ B, and then the update backward of round l - 1 or, after round 0, the
 * gradients of W0 and b0 (dz0 = dh where z0 > 0) */
template <bool FIRST>
__global__ __launch_bounds__(MP_RB, 2) void k_mp_round_bwd(uint32_t N, uint32_t chunk, int l, const float *__restrict__ ideg,
                                                        const unsigned short *__restrict__ wb,
                                                        const float *__restrict__ dP, const float *__restrict__ dQ,
                                                        const float *__restrict__ Hl, const float *__restrict__ ZU,
                                                        const float *__restrict__ H, const float *__restrict__ M,
                                                        float *__restrict__ dhn, float *__restrict__ dm,
                                                        float *__restrict__ part)
{
  __shared__ __align__(16) unsigned char lds[MP_BWD_LDS];
  short *T = reinterpret_cast<short *>(lds) + (threadIdx.x >> 6) * MP_BWD_TILES;
  float *sh = reinterpret_cast<float *>(lds);
  const uint32_t li = threadIdx.x & 31u, h4 = (threadIdx.x & 32u) >> 3;
  const uint32_t p = kf_xcd_block(), n0 = p * chunk, n1 = min(N, n0 + chunk);
  f32x16 ga = mp_zero(), gb = mp_zero(), gu = mp_zero(), gw = mp_zero();
  float bu[16];
#pragma unroll
  for (int r = 0; r < 16; r++) bu[r] = 0.0f;
  for (uint32_t row = n0 + 32 * (threadIdx.x >> 6); row < n1; row += 32 * MP_TW) {
    const uint32_t v = min(row + li, n1 - 1);
    const bool on = row + li < n1;
    float x[16], y[16], h[16], dh[16];
    mp_row_ld(dP, v, x);
    mp_row_ld(dQ, v, y);
    mp_row_ld(Hl, v, h);
    mp_row_ld(dhn, v, dh);
    wave_lds_sync();
    f32x16 acc = mp_mm<4, 2 * MP_H>(wb + MPB_ABT(l), 0, x, mp_zero());
    acc = mp_mm<4, 2 * MP_H>(wb + MPB_ABT(l), MP_H, y, acc);
#pragma unroll
    for (int r = 0; r < 16; r++) {
      x[r] = on ? x[r] : 0.0f;
      y[r] = on ? y[r] : 0.0f;
    }
    mp_tile_put<4>(T, x);
    mp_tile_put<4>(T + 32 * MP_TS, y);
    mp_tile_put<4>(T + 64 * MP_TS, h);
    mp_bias(acc, NULL, x);
#pragma unroll
    for (int r = 0; r < 16; r++) dh[r] = dh[r] + x[r];
    wave_lds_sync();
    ga = mp_tile_mm<32, 32>(T, T + 64 * MP_TS, ga);
    gb = mp_tile_mm<32, 32>(T + 32 * MP_TS, T + 64 * MP_TS, gb);
    if (!FIRST) {
      mp_update_bwd(dh, v, on, ZU, H, M, wb + MPB_UT(l - 1), wb + MPB_VT(l - 1), ideg[v], dhn, dm, T, bu, gu, gw);
    } else {
      /* ZU is z0, H the features (16 per vertex) */
      mp_row_ld(ZU, v, x);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        x[r] = on && x[r] > 0.0f ? dh[r] : 0.0f;
        bu[r] += x[r];
      }
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const float4 t = *reinterpret_cast<const float4 *>(H + (size_t)v * MP_NIN + 8 * q + h4);
        y[4 * q] = t.x; y[4 * q + 1] = t.y; y[4 * q + 2] = t.z; y[4 * q + 3] = t.w;
      }
      wave_lds_sync();
      mp_tile_put<4>(T, x);
      mp_tile_put<2>(T + 32 * MP_TS, y);
      wave_lds_sync();
      gu = mp_tile_mm<32, MP_NIN>(T, T + 32 * MP_TS, gu);
    }
  }
  float *pp = part + (size_t)p * MP_NPARAM;
  mp_wsum<MP_H, MP_H>(ga, sh, pp + MP_A(l));
  mp_wsum<MP_H, MP_H>(gb, sh, pp + MP_B(l));
  if (!FIRST) {
    mp_wsum<MP_H, MP_H>(gu, sh, pp + MP_U(l - 1));
    mp_wsum<MP_H, MP_H>(gw, sh, pp + MP_V(l - 1));
    mp_bsum(bu, sh, pp + MP_UB(l - 1));
  } else {
    mp_wsum<MP_H, MP_NIN>(gu, sh, pp + MP_W0);
    mp_bsum(bu, sh, pp + MP_B0);
  }
}

/* ---- loss ---------------------------------------------------------------------------- */

/* The residual y the loss is formed of and, per workgroup, its sum of squares
 * and the reference's: METRIC 0 y = e against |target|, 1 y = A e against |v|,
 * 2 y = A e - v against |v|.  A quad of lanes per block row, lane c forming
 * component c (as spmv.hip): the quad reads a whole 64-byte block at once,
 * where one lane per row read 64 rows' blocks side by side (331,776 vertices:
 * 91 us against 120 us for the product alone and 20 us for the rest). */
template <int METRIC>
__global__ __launch_bounds__(MP_RB) void k_mp_resid(uint32_t N, const uint32_t *__restrict__ rowptr,
                                                    const uint32_t *__restrict__ col, const float *__restrict__ A,
                                                    const float *__restrict__ e, const double *__restrict__ ref,
                                                    float *__restrict__ y, double2 *__restrict__ lpart)
{
  __shared__ double sh[2 * MP_RB / 64];
  const uint32_t i = kf_xcd_block() * (MP_RB / 4) + (threadIdx.x >> 2), c = threadIdx.x & 3u;
  double s = 0.0, t = 0.0;
  if (i < N) {
    const size_t o = 4 * (size_t)i + c;
    float a;
    if (METRIC == 0) {
      a = e[o];
    } else {
      a = 0.0f;
      const uint32_t j0 = rowptr[i], j1 = rowptr[i + 1];
      for (uint32_t j = j0; j < j1; j += 4) {
        float4 b[4], x[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const uint32_t k = min(j + q, j1 - 1);
          b[q] = *(const float4 *)(A + 16 * (size_t)k + 4 * c);
          x[q] = *(const float4 *)(e + 4 * (size_t)col[k]);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float r = a + (b[q].x * x[q].x + b[q].y * x[q].y + b[q].z * x[q].z + b[q].w * x[q].w);
          a = j + q < j1 ? r : a;
        }
      }
      if (METRIC == 2) a = (float)((double)a - ref[o]);
      y[o] = a;
    }
    s = (double)a * (double)a;
    t = ref[o] * ref[o];
  }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    s += __shfl_xor(s, m, 64);
    t += __shfl_xor(t, m, 64);
  }
  if ((threadIdx.x & 63u) == 0) {
    sh[2 * (threadIdx.x >> 6)] = s;
    sh[2 * (threadIdx.x >> 6) + 1] = t;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < MP_RB / 64; w++) {
      s += sh[2 * w];
      t += sh[2 * w + 1];
    }
    lpart[kf_xcd_block()] = make_double2(s, t);
  }
}

/* loss = sum of the residual's partials / sum of the reference's into out[0];
 * the gradient scale 2 / the reference sum into sc[3] (one workgroup, each
 * thread every 1024th partial, then a fixed tree; one lane walking them took
 * 99 us) */
__global__ __launch_bounds__(1024) void k_mp_loss_finish(const double2 *__restrict__ lpart, uint32_t nb,
                                                         float *__restrict__ out, float *__restrict__ sc)
{
  __shared__ double sa[1024], st[1024];
  const uint32_t i = threadIdx.x;
  double a = 0.0, t = 0.0;
  for (uint32_t b = i; b < nb; b += 1024) {
    a += lpart[b].x;
    t += lpart[b].y;
  }
  sa[i] = a;
  st[i] = t;
  __syncthreads();
  for (uint32_t s = 512; s > 0; s >>= 1) {
    if (i < s) {
      sa[i] += sa[i + s];
      st[i] += st[i + s];
    }
    __syncthreads();
  }
  if (i == 0) {
    a = sa[0];
    t = st[0];
    out[0] = t > 0.0 ? (float)(a / t) : 0.0f;
    sc[3] = t > 0.0 ? (float)(2.0 / t) : 0.0f;
  }
}

/* g = sc[3] A^T y (TRANS; y for METRIC 0): g_j sums A(i, j)^T y_i over row
 * j's positions k (column i = col[k], A(i, j) at tpos[k]; the pattern is
 * structurally symmetric).  A quad of lanes per row, lane c reading column c
 * of the blocks: four 16-byte runs a block (331,776 vertices: 107 us against
 * 166 us with a lane per row, and a pass for the scale). */
template <bool TRANS>
__global__ __launch_bounds__(MP_RB) void k_mp_loss_grad(uint32_t N, const uint32_t *__restrict__ rowptr,
                                                        const uint32_t *__restrict__ col,
                                                        const uint32_t *__restrict__ tpos, const float *__restrict__ A,
                                                        const float *__restrict__ y, const float *__restrict__ sc,
                                                        float *__restrict__ g)
{
  const uint32_t i = kf_xcd_block() * (MP_RB / 4) + (threadIdx.x >> 2), c = threadIdx.x & 3u;
  if (i >= N) return;
  const size_t o = 4 * (size_t)i + c;
  float a;
  if (!TRANS) {
    a = y[o];
  } else {
    a = 0.0f;
    const uint32_t j0 = rowptr[i], j1 = rowptr[i + 1];
    for (uint32_t j = j0; j < j1; j += 4) {
      float4 x[4];
      float b[4][4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint32_t k = min(j + q, j1 - 1);
        const float *p = A + 16 * (size_t)tpos[k] + c;
#pragma unroll
        for (int r = 0; r < 4; r++) b[q][r] = p[4 * r];
        x[q] = *(const float4 *)(y + 4 * (size_t)col[k]);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float r = a + (b[q][0] * x[q].x + b[q][1] * x[q].y + b[q][2] * x[q].z + b[q][3] * x[q].w);
        a = j + q < j1 ? r : a;
      }
    }
  }
  g[o] = a * sc[3];
}

/* A (FP64 or FP32 BSR values) as FP32 */
template <typename TA>
__global__ __launch_bounds__(MP_RB) void k_mp_to_f32(size_t n, const TA *__restrict__ a, float *__restrict__ out)
{
  const size_t k = (size_t)blockIdx.x * MP_RB + threadIdx.x;
  if (k < n) out[k] = (float)a[k];
}

/* ---- Adam ---------------------------------------------------------------------- */

/* One block: global gradient norm (fixed tree), clip to gclip (<= 0: none),
 * then m = b1 m + (1-b1) g, v = b2 v + (1-b2) g^2,
 * theta -= lr (m c1) / (sqrt(v c2) + eps), c1 = 1/(1-b1^t), c2 = 1/(1-b2^t). */
__global__ __launch_bounds__(1024) void k_mp_adam(float *__restrict__ theta, float *__restrict__ m,
                                                  float *__restrict__ v, const float *__restrict__ grad, float lr,
                                                  float b1, float b2, float eps, float c1, float c2, float gclip,
                                                  float *__restrict__ gnorm_out)
{
  __shared__ double sh[1024];
  const int t = threadIdx.x;
  double acc = 0.0;
  for (int i = t; i < MP_NPARAM; i += 1024) acc += (double)grad[i] * (double)grad[i];
  sh[t] = acc;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if (t < s) sh[t] += sh[t + s];
    __syncthreads();
  }
  const double gn = sqrt(sh[0]);
  const float scale = (gclip > 0.0f && gn > (double)gclip) ? (float)((double)gclip / gn) : 1.0f;
  if (t == 0 && gnorm_out) *gnorm_out = (float)gn;
  for (int i = t; i < MP_NPARAM; i += 1024) {
    const float g = grad[i] * scale;
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * (g * g);
    m[i] = mi;
    v[i] = vi;
    theta[i] = theta[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  }
}

/* bf16 copies of the dense weights (forward and transposed) */
__global__ void k_mp_pack(const float *__restrict__ theta, unsigned short *__restrict__ wb)
{
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= MPB_SIZE) return;
  float w = 0.0f;
  const uint32_t HH = MP_H * MP_H;
  if (t < MPB_A(0)) {
    w = theta[MP_W0 + t]; /* 32 x 16 as stored */
  } else if (t < MPB_WSA) {
    const uint32_t r = t - MPB_A(0), l = r / (4 * HH), q = r % (4 * HH);
    if (q < HH) w = theta[MP_A(l) + q];
    else if (q < 2 * HH) w = theta[MP_B(l) + q - HH];
    else {
      const uint32_t qq = q - 2 * HH, o = qq / (2 * MP_H), k = qq % (2 * MP_H);
      w = k < MP_H ? theta[MP_U(l) + o * MP_H + k] : theta[MP_V(l) + o * MP_H + (k - MP_H)];
    }
  } else if (t < MPB_WB) {
    w = theta[MP_WSA + (t - MPB_WSA)];
  } else if (t < MPB_FWD) {
    const uint32_t q = t - MPB_WB, o = q / MP_H, k = q % MP_H;
    w = o < 16 ? theta[MP_WB + o * MP_H + k] : 0.0f;
  } else if (t < MPB_HT) {
    const uint32_t r = t - MPB_FWD, l = r / (4 * HH), q = r % (4 * HH);
    if (q < 2 * HH) {
      /* U^T then V^T: row o, column k = U[k][o] (V[k][o]) */
      const uint32_t which = q / HH, qq = q % HH, o = qq / MP_H, k = qq % MP_H;
      w = theta[(which ? MP_V(l) : MP_U(l)) + k * MP_H + o];
    } else {
      const uint32_t qq = q - 2 * HH, o = qq / (2 * MP_H), k = qq % (2 * MP_H);
      w = k < MP_H ? theta[MP_A(l) + k * MP_H + o] : theta[MP_B(l) + (k - MP_H) * MP_H + o];
    }
  } else {
    /* [WSA^T Wb^T]: row o (hidden channel), column k < 32: WSA[k][o], then Wb[k - 32][o] */
    const uint32_t q = t - MPB_HT, o = q / (2 * MP_H), k = q % (2 * MP_H);
    if (k < MP_H) w = theta[MP_WSA + k * MP_H + o];
    else if (k - MP_H < 16) w = theta[MP_WB + (k - MP_H) * MP_H + o];
  }
  wb[t] = f2bf(w);
}

/* ---- the network object ------------------------------------------------------------ */

struct kf_mpnn {
  kf_ctx *c;
  uint32_t N, nparts, chunk, nslot, nvblk, nlblk;   /* blocks of vertices, of block rows by quads */
  float *theta, *am, *av, *grad, *part, *sc, *gnorm, *losses;
  uint32_t nloss_cap, nloss;
  unsigned short *wb;
  float4 *ev;
  float *X, *Z0, *H[MP_NR + 1], *P[MP_NR], *Q[MP_NR], *M[MP_NR], *ZU[MP_NR];
  uint32_t *pos[MP_NR];      /* per round: which messages were positive (k_mp_message) */
  uint32_t words;            /* ... words per vertex and lane */
  float *OP1, *OPQ;          /* operator coefficients of the prepared slot */
  float *dhn, *dm, *dP, *dQ; /* backward: d h before the messages' part, d m / deg, d P, d Q */
  float *ideg;               /* 1 / max(degree, 1) */
  float *dstore, *isd;       /* per slot: FP32 [N][16] diagonal blocks, 1 / their RMS */
  double *red;
  double2 *lpart;
  float *ebuf, *ybuf, *gbuf; /* loss: error, A error, gradient (N x 4) */
  float **mslot;             /* per slot: the assembled Jacobian (FP32 BSR) or NULL */
  uint32_t *tpos;            /* BSR position of the transposed block */
  int t;                     /* Adam steps so far */
  int metric;                /* loss: 0 |e|^2/|target|^2, 1 |A e|^2/|v|^2,
                                2 |A (base + G base) - v|^2/|v|^2 */
  int prepared;              /* slot whose operator OP1/OPQ hold, -1: none */
};

template <typename T>
static T *mp_alloc(size_t n)
{
  void *p = NULL;
  KF_CHECK(hipMalloc(&p, (n ? n : 1) * sizeof(T)));
  return (T *)p;
}

static void mp_check_slot(const kf_mpnn *net, int slot)
{
  if (slot < 0 || (uint32_t)slot >= net->nslot) {
    fprintf(stderr, "kf: network slot %d out of range [0, %u)\n", slot, net->nslot);
    abort();
  }
}

static void mp_repack(kf_mpnn *net)
{
  hipLaunchKernelGGL(k_mp_pack, dim3(kf_blocks_for(MPB_SIZE, 256)), dim3(256), 0, net->c->stream, net->theta,
                     net->wb);
  KF_LAUNCH_CHECK();
  net->prepared = -1;
}

/* the context network on slot `slot`'s diagonal blocks and the operator
 * coefficients OP1, OPQ; every activation stays in the object for backward */
static void mp_context(kf_mpnn *net, int slot)
{
  kf_ctx *c = net->c;
  hipStream_t st = c->stream;
  const uint32_t N = net->N, nt = kf_blocks_for(N, 32 * MP_TW);
  const float *th = net->theta, *nf = NULL;
  const unsigned short *wb = net->wb;
  hipLaunchKernelGGL(k_mp_in, dim3(nt), dim3(MP_RB), 0, st, N, net->dstore + (size_t)slot * 16 * N, net->isd + slot, wb,
                     th, net->X, net->Z0, net->H[0], net->P[0], net->Q[0]);
  for (int l = 0; l < MP_NR; l++) {
    const bool last = l == MP_NR - 1;
    hipLaunchKernelGGL(k_mp_message, dim3(kf_blocks_for(N, MP_VW)), dim3(MP_RB), 0, st, c->d, net->ev, net->P[l],
                       net->Q[l], th, (uint32_t)MP_C(l), (uint32_t)MP_CB(l), net->M[l], net->pos[l], net->words);
    hipLaunchKernelGGL(k_mp_update, dim3(nt), dim3(MP_RB), 0, st, N, net->H[l], net->M[l], wb + MPB_UV(l),
                       th + MP_UB(l), wb + (last ? MPB_WSA : MPB_A(l + 1)), last ? th + MP_BSA : nf,
                       wb + (last ? MPB_WB : MPB_B(l + 1)), net->ZU[l], net->H[l + 1], last ? net->OP1 : net->P[l + 1],
                       last ? net->OPQ : net->Q[l + 1]);
  }
  KF_LAUNCH_CHECK();
  net->prepared = slot;
}

/* loss of (v, base, target) and the parameter gradient into net->grad; the
 * loss lands in *loss_dev */
static void mp_loss_grad(kf_mpnn *net, int slot, const double *v, const double *base, const double *target,
                         float *loss_dev)
{
  kf_ctx *c = net->c;
  hipStream_t st = c->stream;
  const uint32_t N = net->N, P = net->nparts, ch = net->chunk, nb = net->nlblk;
  const float *nf = NULL;
  const int metric = net->metric;
  const float *A = net->mslot[slot];
  if (metric >= 1 && !A) {
    fprintf(stderr, "kf: the A-norm loss needs the Jacobian of slot %d (kf_mpnn_take_matrix)\n", slot);
    abort();
  }
  mp_context(net, slot);
  hipLaunchKernelGGL(k_mp_apply, dim3(net->nvblk), dim3(MP_RB), 0, st, c->d, net->ev, net->OP1, net->OPQ, net->theta,
                     base, (double *)NULL, 0, metric == 2 ? NULL : target, net->ebuf);
#define MP_RESID(METRIC, REF)                                                                                      \
  hipLaunchKernelGGL(k_mp_resid<METRIC>, dim3(nb), dim3(MP_RB), 0, st, N, c->d.rowptr, c->d.col, A, net->ebuf, REF, \
                     net->ybuf, net->lpart)
  if (metric == 0) MP_RESID(0, target);
  else if (metric == 1) MP_RESID(1, v);
  else MP_RESID(2, v);
#undef MP_RESID
  hipLaunchKernelGGL(k_mp_loss_finish, dim3(1), dim3(1024), 0, st, net->lpart, nb, loss_dev, net->sc);
  if (metric == 0)
    hipLaunchKernelGGL(k_mp_loss_grad<false>, dim3(nb), dim3(MP_RB), 0, st, N, c->d.rowptr, c->d.col, net->tpos, A,
                       net->ebuf, net->sc, net->gbuf);
  else
    hipLaunchKernelGGL(k_mp_loss_grad<true>, dim3(nb), dim3(MP_RB), 0, st, N, c->d.rowptr, c->d.col, net->tpos, A,
                       net->ybuf, net->sc, net->gbuf);
  const int L = MP_NR - 1;
  hipLaunchKernelGGL(k_mp_head_bwd, dim3(P), dim3(MP_RB), 0, st, c->d, ch, net->ev, net->ideg, base, net->gbuf, net->wb,
                     net->H[MP_NR], net->ZU[L], net->H[L], net->M[L], net->dhn, net->dm, net->part);
  for (int l = L; l >= 0; l--) {
    hipLaunchKernelGGL(k_mp_message_bwd, dim3(P), dim3(MP_RB), 0, st, c->d, ch, net->ev, net->pos[l], net->words,
                       net->dm, (uint32_t)MP_C(l), (uint32_t)MP_CB(l), net->dP, net->dQ, net->part);
    if (l > 0)
      hipLaunchKernelGGL(k_mp_round_bwd<false>, dim3(P), dim3(MP_RB), 0, st, N, ch, l, net->ideg, net->wb, net->dP,
                         net->dQ, net->H[l], net->ZU[l - 1], net->H[l - 1], net->M[l - 1], net->dhn, net->dm, net->part);
    else
      hipLaunchKernelGGL(k_mp_round_bwd<true>, dim3(P), dim3(MP_RB), 0, st, N, ch, l, net->ideg, net->wb, net->dP,
                         net->dQ, net->H[0], net->Z0, net->X, nf, net->dhn, (float *)NULL, net->part);
  }
  hipLaunchKernelGGL(k_mp_grad_reduce, dim3(kf_blocks_for(MP_NPARAM, 64)), dim3(1024), 0, st, net->part, P, net->grad);
  KF_LAUNCH_CHECK();
}

/* Initial parameters: normals scaled by sqrt(2 / fan-in) for W0, A, B, C,
 * U and V (U and V halved), zero biases, zero operator heads (G = 0, so
 * training starts from ILU(0) itself).  Normals from splitmix64 and the
 * Box-Muller cosine branch. */
static uint64_t mp_mix(uint64_t *s)
{
  uint64_t z = (*s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

static double mp_normal(uint64_t *s)
{
  const double u1 = ((double)(mp_mix(s) >> 11) + 1.0) * 0x1.0p-53, u2 = (double)(mp_mix(s) >> 11) * 0x1.0p-53;
  return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

extern "C" void kf_mpnn_init_params(float *theta, uint64_t seed)
{
  uint64_t st = seed * 0xD1B54A32D192ED03ull + 1;
  memset(theta, 0, sizeof(float) * MP_NPARAM);
  auto fill = [&](int off, int n, int fan_in, double scale) {
    const double sd = sqrt(2.0 / fan_in) * scale;
    for (int i = 0; i < n; i++) theta[off + i] = (float)(mp_normal(&st) * sd);
  };
  fill(MP_W0, MP_H * MP_NIN, MP_NIN, 1.0);
  for (int l = 0; l < MP_NR; l++) {
    fill(MP_A(l), MP_H * MP_H, MP_H, 1.0);
    fill(MP_B(l), MP_H * MP_H, MP_H, 1.0);
    fill(MP_C(l), MP_H * 3, 3, 1.0);
    fill(MP_U(l), MP_H * MP_H, MP_H, 0.5);
    fill(MP_V(l), MP_H * MP_H, MP_H, 0.5);
  }
}

extern "C" size_t kf_mpnn_nparam(void) { return MP_NPARAM; }
extern "C" size_t kf_mpnn_nhead(void) { return MP_HEADS; }

extern "C" void kf_mpnn_set_params(kf_mpnn *net, const float *theta_host);

extern "C" kf_mpnn *kf_mpnn_create(GEOMETRY *g, const float *theta_host, int nslot)
{
  kf_ctx *c = kf_ctx_of(g);
  if (!theta_host || nslot < 1) {
    fprintf(stderr, "kf: kf_mpnn_create needs initial parameters and at least one slot\n");
    abort();
  }
  kf_mpnn *net = new kf_mpnn();
  memset((void *)net, 0, sizeof(*net));
  net->c = c;
  net->metric = 2;
  net->prepared = -1;
  const uint32_t N = c->d.N;
  net->N = N;
  net->nslot = (uint32_t)nslot;
  uint32_t ch = (N + MP_PARTS - 1) / MP_PARTS;
  ch = ((ch + 31u) / 32u) * 32u;   /* whole tiles of 32 vertices */
  net->chunk = ch;
  net->nparts = (N + ch - 1) / ch;
  net->nvblk = kf_blocks_for(N, MP_RB);
  net->nlblk = kf_blocks_for(N, MP_RB / 4);
  net->theta = mp_alloc<float>(MP_NPARAM);
  net->am = mp_alloc<float>(MP_NPARAM);
  net->av = mp_alloc<float>(MP_NPARAM);
  net->grad = mp_alloc<float>(MP_NPARAM);
  net->part = mp_alloc<float>((size_t)net->nparts * MP_NPARAM);
  net->sc = mp_alloc<float>(8);
  net->gnorm = mp_alloc<float>(1);
  net->nloss_cap = 1u << 16;
  net->losses = mp_alloc<float>(net->nloss_cap);
  net->wb = mp_alloc<unsigned short>(MPB_SIZE);
  /* sliced-ELL slots: the last slice pointer counts them (in units of 64) */
  uint32_t nsl_ent = 0;
  KF_CHECK(hipMemcpy(&nsl_ent, c->d.sell_ptr + c->d.nslice, sizeof(uint32_t), hipMemcpyDeviceToHost));
  net->ev = mp_alloc<float4>((size_t)nsl_ent * 64u);
  const size_t NH = (size_t)N * MP_H;
  net->words = (c->maxrow + 7) / 8;   /* a vertex's edges are its row's off-diagonal blocks, at most maxrow - 1 */
  net->X = mp_alloc<float>((size_t)N * MP_NIN);
  net->Z0 = mp_alloc<float>(NH);
  for (int l = 0; l <= MP_NR; l++) net->H[l] = mp_alloc<float>(NH);
  for (int l = 0; l < MP_NR; l++) {
    net->P[l] = mp_alloc<float>(NH);
    net->Q[l] = mp_alloc<float>(NH);
    net->M[l] = mp_alloc<float>(NH);
    net->ZU[l] = mp_alloc<float>(NH);
    net->pos[l] = mp_alloc<uint32_t>((size_t)N * net->words * 8);
  }
  net->OP1 = mp_alloc<float>(NH);
  net->OPQ = mp_alloc<float>(NH);
  net->dhn = mp_alloc<float>(NH);
  net->dm = mp_alloc<float>(NH);
  net->dP = mp_alloc<float>(NH);
  net->dQ = mp_alloc<float>(NH);
  net->ideg = mp_alloc<float>(N);
  net->dstore = mp_alloc<float>((size_t)nslot * 16 * N);
  net->isd = mp_alloc<float>(nslot);
  net->red = mp_alloc<double>(KF_NRED);
  net->lpart = mp_alloc<double2>(net->nlblk);
  net->ebuf = mp_alloc<float>(4 * (size_t)N);
  net->ybuf = mp_alloc<float>(4 * (size_t)N);
  net->gbuf = mp_alloc<float>(4 * (size_t)N);
  net->mslot = (float **)calloc((size_t)nslot, sizeof(float *));
  if (!net->mslot) abort();
  {
    /* transposed-block positions: (i, j) at k  ->  (j, i) */
    const size_t nnzb = c->nnzb;
    uint32_t *rp = (uint32_t *)malloc(sizeof(uint32_t) * (N + 1)), *cl = (uint32_t *)malloc(sizeof(uint32_t) * nnzb);
    uint32_t *tp = (uint32_t *)malloc(sizeof(uint32_t) * (nnzb ? nnzb : 1));
    if (!rp || !cl || !tp) abort();
    KF_CHECK(hipMemcpy(rp, c->d.rowptr, sizeof(uint32_t) * (N + 1), hipMemcpyDeviceToHost));
    KF_CHECK(hipMemcpy(cl, c->d.col, sizeof(uint32_t) * nnzb, hipMemcpyDeviceToHost));
    for (uint32_t i = 0; i < N; i++)
      for (uint32_t k = rp[i]; k < rp[i + 1]; k++) {
        const uint32_t j = cl[k];
        uint32_t lo = rp[j], hi = rp[j + 1];
        while (lo < hi) { /* columns of a row are sorted */
          const uint32_t mid = (lo + hi) / 2;
          if (cl[mid] < i) lo = mid + 1;
          else hi = mid;
        }
        if (lo == rp[j + 1] || cl[lo] != i) {
          fprintf(stderr, "kf: block pattern is not structurally symmetric\n");
          abort();
        }
        tp[k] = lo;
      }
    net->tpos = mp_alloc<uint32_t>(nnzb ? nnzb : 1);
    KF_CHECK(hipMemcpy(net->tpos, tp, sizeof(uint32_t) * nnzb, hipMemcpyHostToDevice));
    free(rp);
    free(cl);
    free(tp);
  }
  KF_CHECK(hipMemsetAsync(net->dstore, 0, sizeof(float) * (size_t)nslot * 16 * N, c->stream));
  float *ones = (float *)malloc(sizeof(float) * nslot);
  for (int i = 0; i < nslot; i++) ones[i] = 1.0f;
  KF_CHECK(hipMemcpyAsync(net->isd, ones, sizeof(float) * nslot, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_mp_edge_vectors, dim3(kf_blocks_for(N, MP_RB)), dim3(MP_RB), 0, c->stream, c->d, net->ev,
                     net->ideg);
  KF_LAUNCH_CHECK();
  KF_CHECK(hipStreamSynchronize(c->stream));
  free(ones);
  kf_mpnn_set_params(net, theta_host);
  return net;
}

extern "C" void kf_mpnn_set_params(kf_mpnn *net, const float *theta_host)
{
  hipStream_t st = net->c->stream;
  KF_CHECK(hipMemcpyAsync(net->theta, theta_host, sizeof(float) * MP_NPARAM, hipMemcpyHostToDevice, st));
  KF_CHECK(hipMemsetAsync(net->am, 0, sizeof(float) * MP_NPARAM, st));
  KF_CHECK(hipMemsetAsync(net->av, 0, sizeof(float) * MP_NPARAM, st));
  net->t = 0;
  mp_repack(net);
  KF_CHECK(hipStreamSynchronize(st));
}

extern "C" void kf_mpnn_get_params(const kf_mpnn *net, float *theta_host)
{
  KF_CHECK(hipStreamSynchronize(net->c->stream));
  KF_CHECK(hipMemcpy(theta_host, net->theta, sizeof(float) * MP_NPARAM, hipMemcpyDeviceToHost));
}

extern "C" void kf_mpnn_destroy(kf_mpnn *net)
{
  if (!net) return;
  KF_CHECK(hipStreamSynchronize(net->c->stream));
  void *bufs[] = {net->theta, net->am,   net->av,   net->grad,  net->part, net->sc,   net->gnorm, net->losses,
                  net->wb,    net->ev,   net->X,    net->Z0,    net->OP1,  net->OPQ,  net->ideg,  net->dhn,
                  net->dm,    net->dP,   net->dQ,   net->dstore,
                  net->isd,   net->red,  net->lpart, net->ebuf, net->ybuf,  net->gbuf,
                  net->tpos};
  for (void *p : bufs)
    if (p) KF_CHECK(hipFree(p));
  for (uint32_t k = 0; k < net->nslot; k++)
    if (net->mslot[k]) KF_CHECK(hipFree(net->mslot[k]));
  free(net->mslot);
  for (int l = 0; l <= MP_NR; l++) KF_CHECK(hipFree(net->H[l]));
  for (int l = 0; l < MP_NR; l++) {
    KF_CHECK(hipFree(net->P[l]));
    KF_CHECK(hipFree(net->Q[l]));
    KF_CHECK(hipFree(net->M[l]));
    KF_CHECK(hipFree(net->ZU[l]));
    KF_CHECK(hipFree(net->pos[l]));
  }
  delete net;
}

/* the current ILU factor's diagonal blocks (and 1 / their RMS) into `slot` */
extern "C" void kf_mpnn_take_diag(kf_mpnn *net, int slot)
{
  mp_check_slot(net, slot);
  kf_ctx *c = net->c;
  hipStream_t st = c->stream;
  const uint32_t N = net->N;
  float *D = net->dstore + (size_t)slot * 16 * N;
  const uint32_t nb = kf_blocks_for(16 * (size_t)N, MP_RB);
  if (c->opt.prec == KF_PREC_FP64)
    hipLaunchKernelGGL(k_mp_take_diag<double>, dim3(nb), dim3(MP_RB), 0, st, N, c->d.diag, (const double *)c->a64, D);
  else
    hipLaunchKernelGGL(k_mp_take_diag<float>, dim3(nb), dim3(MP_RB), 0, st, N, c->d.diag, (const float *)c->a32, D);
  hipLaunchKernelGGL(k_mp_sumsq<float>, dim3(KF_NRED), dim3(MP_RB), 0, st, 16 * (size_t)N, (const float *)D,
                     net->red);
  hipLaunchKernelGGL(k_mp_finish, dim3(1), dim3(MP_RB), 0, st, net->red, 16.0 * N, net->isd + slot);
  KF_LAUNCH_CHECK();
  if (net->prepared == slot) net->prepared = -1;
}

/* the assembled Jacobian (after ComputeA, before ComputeNumericalILU
 * factors it in place) into `slot`, as FP32 */
extern "C" void kf_mpnn_take_matrix(kf_mpnn *net, int slot)
{
  mp_check_slot(net, slot);
  kf_ctx *c = net->c;
  const size_t n = 16 * c->nnzb;
  if (!net->mslot[slot]) net->mslot[slot] = mp_alloc<float>(n);
  if (c->opt.prec == KF_PREC_FP64)
    hipLaunchKernelGGL(k_mp_to_f32<double>, dim3(kf_blocks_for(n, MP_RB)), dim3(MP_RB), 0, c->stream, n,
                       (const double *)c->a64, net->mslot[slot]);
  else
    KF_CHECK(hipMemcpyAsync(net->mslot[slot], c->a32, n * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
  KF_LAUNCH_CHECK();
}

/* 0: |e|^2 / |target|^2;  1: |A e|^2 / |v|^2 with the slot's A;
 * 2 (default): |A (base + G base) - v|^2 / |v|^2 (the target is not read) */
extern "C" void kf_mpnn_set_loss(kf_mpnn *net, int metric)
{
  if (metric < 0 || metric > 2) {
    fprintf(stderr, "kf: kf_mpnn_set_loss: no loss %d\n", metric);
    abort();
  }
  net->metric = metric;
}

/* diagonal blocks given by the caller (host FP64 [N][16]) into `slot` */
extern "C" void kf_mpnn_set_diag(kf_mpnn *net, int slot, const double *D_host)
{
  mp_check_slot(net, slot);
  kf_ctx *c = net->c;
  const size_t n = 16 * (size_t)net->N;
  float *tmp = (float *)malloc(sizeof(float) * n);
  for (size_t i = 0; i < n; i++) tmp[i] = (float)D_host[i];
  float *D = net->dstore + (size_t)slot * n;
  KF_CHECK(hipMemcpyAsync(D, tmp, sizeof(float) * n, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_mp_sumsq<float>, dim3(KF_NRED), dim3(MP_RB), 0, c->stream, n, (const float *)D, net->red);
  hipLaunchKernelGGL(k_mp_finish, dim3(1), dim3(MP_RB), 0, c->stream, net->red, (double)n, net->isd + slot);
  KF_LAUNCH_CHECK();
  KF_CHECK(hipStreamSynchronize(c->stream));
  free(tmp);
  if (net->prepared == slot) net->prepared = -1;
}

/* the correction operator of `slot` (the context network on its diagonal
 * blocks); kf_mpnn_forward prepares on demand */
extern "C" void kf_mpnn_prepare(kf_mpnn *net, int slot)
{
  mp_check_slot(net, slot);
  mp_context(net, slot);
}

/* out = G z (add = 0) or out += G z (add = 1), z = ILU^-1 v; device vectors
 * of 4N */
extern "C" void kf_mpnn_forward(kf_mpnn *net, int slot, const double *z, double *out, int add)
{
  mp_check_slot(net, slot);
  if (net->prepared != slot) mp_context(net, slot);
  hipLaunchKernelGGL(k_mp_apply, dim3(net->nvblk), dim3(MP_RB), 0, net->c->stream, net->c->d, net->ev, net->OP1,
                     net->OPQ, net->theta, z, out, add, (const double *)NULL, (float *)NULL);
  KF_LAUNCH_CHECK();
}

/* loss of (v, base, target) and its gradient (host FP32 copy when grad_host
 * is given); device vectors of 4N.  Synchronises. */
extern "C" double kf_mpnn_loss_grad(kf_mpnn *net, int slot, const double *v, const double *base, const double *target,
                                    float *grad_host)
{
  mp_check_slot(net, slot);
  mp_loss_grad(net, slot, v, base, target, net->sc + 4);
  float loss;
  KF_CHECK(hipMemcpyAsync(&loss, net->sc + 4, sizeof(float), hipMemcpyDeviceToHost, net->c->stream));
  if (grad_host)
    KF_CHECK(hipMemcpyAsync(grad_host, net->grad, sizeof(float) * MP_NPARAM, hipMemcpyDeviceToHost, net->c->stream));
  KF_CHECK(hipStreamSynchronize(net->c->stream));
  return (double)loss;
}

static void mp_adam(kf_mpnn *net, float lr, float b1, float b2, float eps, float gclip)
{
  net->t++;
  const float c1 = (float)(1.0 / (1.0 - pow((double)b1, net->t)));
  const float c2 = (float)(1.0 / (1.0 - pow((double)b2, net->t)));
  hipLaunchKernelGGL(k_mp_adam, dim3(1), dim3(1024), 0, net->c->stream, net->theta, net->am, net->av, net->grad, lr,
                     b1, b2, eps, c1, c2, gclip, net->gnorm);
  KF_LAUNCH_CHECK();
  mp_repack(net);
}

/* one Adam step with the gradient of the last kf_mpnn_loss_grad */
extern "C" void kf_mpnn_adam(kf_mpnn *net, float lr, float beta1, float beta2, float eps, float gclip)
{
  mp_adam(net, lr, beta1, beta2, eps, gclip);
  KF_CHECK(hipStreamSynchronize(net->c->stream));
}

/* loss + gradient + Adam (0.9, 0.999, 1e-8) on one pair, queued on the
 * stream with no host round trip; the loss goes to the loss log */
extern "C" void kf_mpnn_train_step(kf_mpnn *net, int slot, const double *v, const double *base, const double *target,
                                   float lr, float gclip)
{
  mp_check_slot(net, slot);
  float *ld = net->losses + (net->nloss % net->nloss_cap);
  net->nloss++;
  mp_loss_grad(net, slot, v, base, target, ld);
  mp_adam(net, lr, 0.9f, 0.999f, 1e-8f, gclip);
}

/* the loss log: returns the steps logged since the last reset and copies the
 * first min(cap, 65536) of them */
extern "C" int kf_mpnn_losses(kf_mpnn *net, float *host, int cap)
{
  KF_CHECK(hipStreamSynchronize(net->c->stream));
  const uint32_t n = net->nloss < net->nloss_cap ? net->nloss : net->nloss_cap;
  const uint32_t k = (cap > 0 && (uint32_t)cap < n) ? (uint32_t)cap : n;
  if (k && host) KF_CHECK(hipMemcpy(host, net->losses, sizeof(float) * k, hipMemcpyDeviceToHost));
  return (int)net->nloss;
}

extern "C" void kf_mpnn_reset_losses(kf_mpnn *net) { net->nloss = 0; }

/* activations of the last context pass, for tests: 0 x (N x 16), 1 z0, then
 * per round l: 2+5l h_l, 3+5l P, 4+5l Q, 5+5l m, 6+5l zu; 17 the final h,
 * 18 OP1, 19 OPQ (N x 32 each) */
extern "C" void kf_mpnn_activation(kf_mpnn *net, int which, float *host)
{
  KF_CHECK(hipStreamSynchronize(net->c->stream));
  const size_t NH = (size_t)net->N * MP_H;
  const float *src = NULL;
  size_t n = NH;
  if (which == 0) {
    src = net->X;
    n = (size_t)net->N * MP_NIN;
  } else if (which == 1) src = net->Z0;
  else if (which == 17) src = net->H[MP_NR];
  else if (which == 18) src = net->OP1;
  else if (which == 19) src = net->OPQ;
  else if (which >= 2 && which < 17) {
    const int l = (which - 2) / 5, k = (which - 2) % 5;
    const float *tab[5] = {net->H[l], net->P[l], net->Q[l], net->M[l], net->ZU[l]};
    src = tab[k];
  } else {
    fprintf(stderr, "kf: kf_mpnn_activation: no activation %d\n", which);
    abort();
  }
  KF_CHECK(hipMemcpy(host, src, sizeof(float) * n, hipMemcpyDeviceToHost));
}
