/*
 * ilu.hip -- block ILU(0) of the BSR Jacobian, in place: strictly lower
 * blocks become L (unit diagonal implied), upper blocks U, and the diagonal
 * holds inv(U(i,i)), the storage the reference's ilu_Edmond leaves in A
 * (matrix/ilu.cpp:49-138) and its triangular solve expects.
 *
 * The reference's one-thread sweep is sequential ILU(0) in natural row
 * order: for each row i and each column k of its pattern, ascending,
 *   a = A(i,k) - sum_{m < min(i,k)} L(i,m) U(m,k)   (m ascending)
 *   L(i,k) = a inv(U(k,k))  if k < i,   U(i,k) = a  otherwise.
 * Here row i runs on one wavefront as soon as the rows of its lower
 * pattern are final (level schedule of matrix/init.cpp:194-232, sync-free:
 * see sync.h).  The row is staged in LDS; for each lower block m ascending
 * 16 lanes form L(i,m) = a(i,m) inv(U(m,m)) and then 4 x 16 lanes subtract
 * L(i,m) U(m,k) from every matching block of the row, so each block sees
 * its updates in ascending m, in the reference's block-product order
 * (matrix/init.cpp:105-116).  16 lanes then form the cofactor inverse of the
 * diagonal block, one lane per entry, with the expressions of
 * matrix/inverse.cpp:195-352.
 */
#include "sync.h"
#include "handoff.h"

/* matrix/inverse.cpp:200-326: entry e of the adjugate is
 * s0*(a b c) s1*(...) ... six signed triple products summed left to right */
__constant__ uint8_t kf_cof_idx[16][6][3] = {
  {{5, 10, 15}, {5, 11, 14}, {9, 6, 15}, {9, 7, 14}, {13, 6, 11}, {13, 7, 10}},
  {{1, 10, 15}, {1, 11, 14}, {9, 2, 15}, {9, 3, 14}, {13, 2, 11}, {13, 3, 10}},
  {{1, 6, 15}, {1, 7, 14}, {5, 2, 15}, {5, 3, 14}, {13, 2, 7}, {13, 3, 6}},
  {{1, 6, 11}, {1, 7, 10}, {5, 2, 11}, {5, 3, 10}, {9, 2, 7}, {9, 3, 6}},
  {{4, 10, 15}, {4, 11, 14}, {8, 6, 15}, {8, 7, 14}, {12, 6, 11}, {12, 7, 10}},
  {{0, 10, 15}, {0, 11, 14}, {8, 2, 15}, {8, 3, 14}, {12, 2, 11}, {12, 3, 10}},
  {{0, 6, 15}, {0, 7, 14}, {4, 2, 15}, {4, 3, 14}, {12, 2, 7}, {12, 3, 6}},
  {{0, 6, 11}, {0, 7, 10}, {4, 2, 11}, {4, 3, 10}, {8, 2, 7}, {8, 3, 6}},
  {{4, 9, 15}, {4, 11, 13}, {8, 5, 15}, {8, 7, 13}, {12, 5, 11}, {12, 7, 9}},
  {{0, 9, 15}, {0, 11, 13}, {8, 1, 15}, {8, 3, 13}, {12, 1, 11}, {12, 3, 9}},
  {{0, 5, 15}, {0, 7, 13}, {4, 1, 15}, {4, 3, 13}, {12, 1, 7}, {12, 3, 5}},
  {{0, 5, 11}, {0, 7, 9}, {4, 1, 11}, {4, 3, 9}, {8, 1, 7}, {8, 3, 5}},
  {{4, 9, 14}, {4, 10, 13}, {8, 5, 14}, {8, 6, 13}, {12, 5, 10}, {12, 6, 9}},
  {{0, 9, 14}, {0, 10, 13}, {8, 1, 14}, {8, 2, 13}, {12, 1, 10}, {12, 2, 9}},
  {{0, 5, 14}, {0, 6, 13}, {4, 1, 14}, {4, 2, 13}, {12, 1, 6}, {12, 2, 5}},
  {{0, 5, 10}, {0, 6, 9}, {4, 1, 10}, {4, 2, 9}, {8, 1, 6}, {8, 2, 5}}};
/* bit t set: term t is subtracted (term 0: its first factor is negated) */
__constant__ uint8_t kf_cof_neg[16] = {0x26, 0x19, 0x26, 0x19, 0x19, 0x26, 0x19, 0x26,
                                      0x26, 0x19, 0x26, 0x19, 0x19, 0x26, 0x19, 0x26};

#define ILU_MAXROW 128

/* d = A B for 4x4 row-major blocks, entry (r, c) of lane e = 4 r + c, with the
 * reference's summation order (matrix/init.cpp:105-116) */
template <typename T>
__device__ __forceinline__ T blk_mul(const T *A, const T *B, uint32_t r, uint32_t c)
{
  T s = T(0);
#pragma unroll
  for (int k = 0; k < 4; k++) s += A[4 * r + k] * B[4 * k + c];
  return s;
}

/* value of lane I of this lane's quad: a quad holds one row of a 4x4 block,
 * so these are the row's four entries */
template <int I>
__device__ __forceinline__ float quad_bcast(float v)
{
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), I * 0x55, 0xf, 0xf, true));
}

template <int I>
__device__ __forceinline__ double quad_bcast(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), I * 0x55, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), I * 0x55, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

/* blk_mul with the left block in registers (one entry per lane) and column c
 * of the right block in b: the same sum in the same order */
template <typename T>
__device__ __forceinline__ T row_mul(T a, const T b[4])
{
  T s = T(0);
  s += quad_bcast<0>(a) * b[0];
  s += quad_bcast<1>(a) * b[1];
  s += quad_bcast<2>(a) * b[2];
  s += quad_bcast<3>(a) * b[3];
  return s;
}

/* column c of the 4x4 block at p */
template <typename T>
__device__ __forceinline__ void blk_col(const T *p, uint32_t c, T b[4])
{
#pragma unroll
  for (int k = 0; k < 4; k++) b[k] = p[4 * k + c];
}

__device__ __forceinline__ float lane_get(float v, int l)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ double lane_get(double v, int l)
{
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

/* EXACT: the reference's one-thread sweep bit for bit.  Each block it forms
 * ends with the product of the last common pair of its merge (matrix/ilu.cpp:
 * 71-86): subtracted, then added back, which rounds.  For a lower block (i,k)
 * that pair is L_old(i,k) U(k,k), where L_old is what the L copy held before
 * this sweep -- the previous sweep's L(i,k), or, for the first lower slot of
 * row i, the Jacobian block A(i, k_last) that matrix/matrix.cpp:145 copies
 * there during the fill (k_last = the row's largest lower column, the last
 * lower block the fill touches); for an upper block it is I A(i,k).  lold
 * keeps the previous sweep's L blocks (BSR positions), ud the non-inverted
 * U(k,k). */
template <typename T, bool EXACT>
__global__ __launch_bounds__(64) void k_ilu(kf_dv d, const uint32_t *__restrict__ rows, uint32_t nrows,
                                            uint32_t *ticket, uint32_t base, uint32_t *rdone, uint32_t epoch,
                                            T *a, T *lold, T *ud)
{
  __shared__ uint32_t scol[ILU_MAXROW];
  __shared__ T sa[ILU_MAXROW * 16];
  __shared__ T sq[16];
  const uint32_t lane = threadIdx.x;
  const uint32_t e = lane & 15, er = e >> 2, ec = e & 3, grp = lane >> 4;
  bool aborted = false;
  for (;;) {
    const uint32_t t = next_ticket(ticket, base);
    if (t >= nrows) break;
    const uint32_t i = rows[t];
    const uint32_t j0 = d.rowptr[i], j1 = d.rowptr[i + 1], jd = d.diag[i];
    const uint32_t L = j1 - j0, nlow = jd - j0, pd = jd - j0;
    for (uint32_t k = lane; k < L; k += 64) scol[k] = d.col[j0 + k];
    for (uint32_t k = lane; k < 16 * L; k += 64) sa[k] = a[16 * (size_t)j0 + k];
    __syncthreads();
    for (uint32_t k = lane; k < nlow; k += 64) wait_row(rdone, scol[k], epoch, d.err, aborted, d.spin_sleep);
    aborted = __any(aborted);
    consume_fence();
    __syncthreads();

    for (uint32_t p = 0; p < nlow; p++) {
      const uint32_t m = scol[p];
      const T *dm = a + 16 * (size_t)d.diag[m];
      if (EXACT) {
        /* a(i,m) = (a - L_old U(m,m)) + L_old U(m,m) */
        const T *lo = p == 0 ? a + 16 * ((size_t)j0 + nlow - 1) : lold + 16 * ((size_t)j0 + p);
        if (lane < 16) sq[e] = lo[e];
        __syncthreads();
        T dq = T(0);
        if (lane < 16) dq = blk_mul(sq, ud + 16 * (size_t)m, er, ec);
        __syncthreads();
        if (lane < 16) {
          T v = sa[16 * p + e];
          v = T(-1) * dq + v;
          v = T(1) * dq + v;
          sa[16 * p + e] = v;
        }
        __syncthreads();
      }
      /* L(i,m) = a(i,m) inv(U(m,m)) */
      T lv = T(0);
      if (lane < 16) lv = blk_mul(sa + 16 * p, dm, er, ec);
      __syncthreads();
      if (lane < 16) sa[16 * p + e] = lv;
      __syncthreads();
      /* a(i,k) -= L(i,m) U(m,k) for the upper blocks (m,k) of row m in row i */
      const uint32_t m1 = d.rowptr[m + 1];
      for (uint32_t jm = d.diag[m] + 1 + grp; jm < m1; jm += 4) {
        const uint32_t kc = d.col[jm];
        uint32_t lo = 0, hi = L;
        while (lo < hi) {
          const uint32_t mid = (lo + hi) >> 1;
          if (scol[mid] < kc) lo = mid + 1;
          else hi = mid;
        }
        if (lo < L && scol[lo] == kc) {
          const T s = blk_mul(sa + 16 * p, a + 16 * (size_t)jm, er, ec);
          sa[16 * lo + e] = sa[16 * lo + e] - s;
        }
      }
      __syncthreads();
    }

    if (EXACT) {
      /* upper blocks: a = (a - I A(i,k)) + I A(i,k), A = the fill's block */
      for (uint32_t p = pd + grp; p < L; p += 4) {
        const T *a0 = a + 16 * ((size_t)j0 + p);
        T dq = T(0);
#pragma unroll
        for (int k = 0; k < 4; k++) dq += (er == (uint32_t)k ? T(1) : T(0)) * a0[4 * k + ec];
        T v = sa[16 * p + e];
        v = T(-1) * dq + v;
        v = T(1) * dq + v;
        sa[16 * p + e] = v;
      }
      __syncthreads();
      if (lane < 16) ud[16 * (size_t)i + e] = sa[16 * pd + e];
    }

    /* diagonal: cofactor inverse, one lane per entry (lanes 16..63 mirror
     * lanes 0..15 so that the shuffles below read defined values) */
    {
      const T *s = sa + 16 * pd;
      const uint8_t neg = kf_cof_neg[e];
      T acc = s[kf_cof_idx[e][0][0]];
      if (neg & 1u) acc = -acc;
      acc = acc * s[kf_cof_idx[e][0][1]] * s[kf_cof_idx[e][0][2]];
#pragma unroll
      for (int tt = 1; tt < 6; tt++) {
        const T pr = s[kf_cof_idx[e][tt][0]] * s[kf_cof_idx[e][tt][1]] * s[kf_cof_idx[e][tt][2]];
        acc = (neg & (1u << tt)) ? acc - pr : acc + pr;
      }
      const T d0 = __shfl(acc, 0, 16), d4 = __shfl(acc, 4, 16), d8 = __shfl(acc, 8, 16), d12 = __shfl(acc, 12, 16);
      T det = s[0] * d0 + s[1] * d4 + s[2] * d8 + s[3] * d12;
      det = T(1) / det;
      acc *= det;
      __syncthreads();
      if (lane < 16) {
        if (!isfinite((double)acc)) atomicOr(d.err, KF_ERR_NONFINITE_PIVOT);
        sa[16 * pd + e] = acc;
      }
    }
    __syncthreads();
    for (uint32_t k = lane; k < 16 * L; k += 64) a[16 * (size_t)j0 + k] = sa[k];
    if (EXACT)
      for (uint32_t k = lane; k < 16 * nlow; k += 64) lold[16 * (size_t)j0 + k] = sa[k];
    publish_fence();
    __syncthreads();
    if (lane == 0) flag_store(rdone + i, epoch);
  }
}

/* Shared-memory layout of k_ilu_rows, sized on the host from the plan:
 * maxrow blocks per row, maxlow lower blocks per row, maxmatch update pairs
 * per row. */
struct ilu_layout {
  uint32_t sa, sa0, ssrc, smoff, slo, stage, bytes;
  __host__ __device__ ilu_layout(uint32_t maxrow, uint32_t maxlow, uint32_t maxmatch, uint32_t tsize, bool exact)
  {
    uint32_t o = 0;
    auto take = [&o](uint32_t n) { const uint32_t r = o; o += (n + 15u) & ~15u; return r; };
    sa = take(16 * tsize * maxrow);
    sa0 = exact ? take(16 * tsize * maxrow) : 0;
    ssrc = take(4 * ((exact ? 2 : 1) * maxlow + maxmatch));
    smoff = take(4 * (maxlow + 1));
    slo = take(2 * (maxmatch + 8));   /* 8 spare pairs, see the elimination */
    stage = take(16 * tsize * ((exact ? 3 : 1) * maxlow + maxmatch + 8));
    bytes = o;
  }
};

#define ILU_Q 4    /* values per lane per load round before the wait */
#define ILU_GMAX 8 /* wavefronts per workgroup at most */
#define ILU_RING 4 /* batches of tickets a workgroup knows of */

/* The tickets of a workgroup.  One atomic on the launch's counter draws a
 * batch of B consecutive tickets (they serialise at about 12 ns each: with 4
 * to an atomic they bounded the FP32 factors of 2.65M vertices at 8.1 ms, with
 * 8 those take 4.5), and the workgroup's wavefronts take them one by one from
 * LDS, in order and without waiting for one another.  B is the number of
 * wavefronts: more rows of one level to a wavefront take it longer, fewer
 * serialise.  The wavefront that takes the first of batch k
 * draws batch k + 2 (after k + 1 has been stored, so that a workgroup's
 * batches ascend), and stores it once it is back, before it waits for any
 * row: entry k % ILU_RING of the ring is k << 32 | first ticket, `read`
 * counts the tickets taken of it.
 * No wait can deadlock: a wavefront takes its next ticket when the row it
 * holds needs no other row any more, so the oldest unfinished ticket of the
 * launch is held by a running wavefront whose dependences are all finished,
 * and the wavefront that is to store a batch stores it without waiting for a
 * row.  The counter advances by kf_ticket_advance_ring(). */
struct ilu_ring {
  unsigned long long entry[ILU_RING];
  uint32_t read[ILU_RING], head;
};

static inline uint32_t kf_ticket_advance_ring(uint32_t ntask, uint32_t nb, uint32_t B)
{
  return B * ((ntask + B - 1) / B + 2 * nb);
}

template <typename V>
__device__ __forceinline__ V lds_load(V *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename V>
__device__ __forceinline__ void lds_store(V *p, V v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* a row's schedule, the same for the whole wavefront */
struct ilu_row {
  uint32_t i, j0, L, nlow, mbeg, mcnt;
};

/* the end of the pairs of lower block p - 1, from the register that holds
 * moff by lane (its lanes past the row's lower blocks hold the pair count) */
__device__ __forceinline__ uint32_t step_end(uint32_t moreg, const uint32_t *smoff, uint32_t p)
{
  if (p < 64) return __builtin_amdgcn_readlane(moreg, p);
  return __builtin_amdgcn_readfirstlane(smoff[p]);
}

/* k_ilu with the row's schedule precomputed on the host (kf_plan_ilu): a
 * record per ticket, the diagonal position of every row it reads from and
 * the list of update pairs (U(m,k) block, position of k in row i).  The
 * wavefront stages inv(U(m,m)), U(m,m) and the U(m,k) blocks in LDS from the
 * published copies (apub), retrying values that still hold the
 * call's sentinel (handoff.h): no flags, no fences.  The rest runs from
 * LDS; the row then publishes its upper blocks, U(i,i) and diagonal inverse
 * and stores its factors in place.  Arithmetic and its order are those of
 * k_ilu.
 *
 * Bound by rows in flight times the time a wavefront spends on one: the
 * round trip for the published blocks (2.4 us under load), the chain of the
 * elimination and the inverse.  So the next row's record and blocks are
 * loaded while this one computes, what its chain does not need is formed
 * while the published blocks are on their way, and their places are one
 * table, so that all of a lane's loads go out together.  Against a version
 * that took each block's place from one of three tables on its own branch,
 * formed L(i,m) on 16 lanes through LDS and loaded each row when its
 * predecessor was done: FP64 (exact) 2.05 -> 1.62 ms on 331,776 vertices and
 * 12.7 -> 9.9 ms on 2.65M, FP32 1.36 -> 1.11 and 8.1 -> 4.5 ms (with the sweeps'
 * copy stored as well 1.73, 10.8, 1.16 and 4.9). */
/* where a row's factors go beside a: the BF16 copy (TS = uint16_t) and, with
 * Jacobi sweeps, the sweeps' sliced copy (val; layout at k_jac_lower_sl), in
 * TS.  Written from the row in LDS, they cost their own stores; as passes
 * after the factorisation the two read and wrote the factors again (1.12M
 * vertices and seven coarse levels: 1.08 ms of 8.0). */
struct ilu_out {
  uint16_t *abf;
  void *val;
  uint32_t K, nslice;
};

__device__ __forceinline__ void ilu_cvt(double v, double *o) { *o = v; }
__device__ __forceinline__ void ilu_cvt(float v, float *o) { *o = v; }
__device__ __forceinline__ void ilu_cvt(float v, uint16_t *o)   /* round to nearest even */
{
  uint32_t u = __float_as_uint(v);
  u += 0x7FFFu + ((u >> 16) & 1u);
  *o = (uint16_t)(u >> 16);
}

__device__ __forceinline__ void ilu_ld4(const float *p, float x[4])
{
  const float4 v = *reinterpret_cast<const float4 *>(p);
  x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
}
__device__ __forceinline__ void ilu_ld4(const double *p, double x[4])
{
  const double2 u = reinterpret_cast<const double2 *>(p)[0], v = reinterpret_cast<const double2 *>(p)[1];
  x[0] = u.x; x[1] = u.y; x[2] = v.x; x[3] = v.y;
}
__device__ __forceinline__ void ilu_st4(double *p, const double x[4])
{
  reinterpret_cast<double2 *>(p)[0] = make_double2(x[0], x[1]);
  reinterpret_cast<double2 *>(p)[1] = make_double2(x[2], x[3]);
}
__device__ __forceinline__ void ilu_st4(float *p, const float x[4])
{
  *reinterpret_cast<float4 *>(p) = make_float4(x[0], x[1], x[2], x[3]);
}
__device__ __forceinline__ void ilu_st4(uint16_t *p, const uint16_t x[4])
{
  *reinterpret_cast<uint2 *>(p) = make_uint2(x[0] | (uint32_t)x[1] << 16, x[2] | (uint32_t)x[3] << 16);
}

template <typename T, bool EXACT, typename TS>
__global__ __launch_bounds__(64 * ILU_GMAX, sizeof(T) == 8 ? 2 : 4)
void k_ilu_rows(kf_dv d, const uint32_t *__restrict__ rec, uint32_t nrows, uint32_t *ticket, uint32_t base, uint32_t B,
                uint32_t nnzb, T *apub, typename sentinel<T>::bits snt, T *a, T *lold, const uint32_t *__restrict__ ldiag,
                const uint32_t *__restrict__ moff, const uint32_t *__restrict__ mjm, const uint16_t *__restrict__ mlo,
                uint32_t maxrow, uint32_t maxlow, uint32_t maxmatch, ilu_out out)
{
  /* values per lane and staging round: one round covers the 45 (EXACT) or 38
   * blocks of a lattice row */
  constexpr int QB = EXACT ? 12 : 10;
  extern __shared__ __align__(16) unsigned char ilu_lds_all[];
  __shared__ ilu_ring ring;
  const ilu_layout lay(maxrow, maxlow, maxmatch, sizeof(T), EXACT);
  unsigned char *ilu_lds = ilu_lds_all + (size_t)(threadIdx.x >> 6) * lay.bytes;   /* this wave's region */
  T *sa = (T *)(ilu_lds + lay.sa);
  T *sa0 = (T *)(ilu_lds + lay.sa0);
  uint32_t *ssrc = (uint32_t *)(ilu_lds + lay.ssrc);
  uint32_t *smoff = (uint32_t *)(ilu_lds + lay.smoff);
  uint16_t *slo = (uint16_t *)(ilu_lds + lay.slo);
  T *stage = (T *)(ilu_lds + lay.stage);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t e = lane & 15, er = e >> 2, ec = e & 3, grp = lane >> 4;
  bool aborted = false;
  /* the cofactor expression of this lane's entry: 18 factor positions of 4
   * bits and the signs, kept in registers (three words and a byte) */
  uint32_t cof[3];
#pragma unroll
  for (int w = 0; w < 3; w++) {
    cof[w] = 0;
#pragma unroll
    for (int q = 0; q < 6; q++) cof[w] |= (uint32_t)kf_cof_idx[e][2 * w + q / 3][q % 3] << (4 * q);
  }
  const uint32_t neg = kf_cof_neg[e];

  if (threadIdx.x == 0) {
    /* batches 0 and 1, one after the other: a workgroup's batches ascend */
    for (uint32_t k = 0; k < ILU_RING; k++) {
      ring.entry[k] = k < 2 ? (unsigned long long)k << 32 | (atomicAdd(ticket, B) - base) : ~0ull;
      ring.read[k] = k < 2 ? 0u : B;
    }
    ring.head = 0;
  }
  __syncthreads();

  /* the wavefront's next ticket; a drawn batch is in `drawn` until put() */
  uint32_t put_k = 0, drawn = 0;
  auto entry = [&](uint32_t k) -> uint32_t {   /* batch k's first ticket, once it is stored */
    unsigned long long en = lds_load(&ring.entry[k % ILU_RING]);
    for (uint32_t n = 0; (uint32_t)(en >> 32) != k; n++) {
      if (n > KF_SPIN_LIMIT) {
        if (lane == 0) atomicOr(d.err, KF_ERR_SPIN_LIMIT);
        return nrows;
      }
      __builtin_amdgcn_s_sleep(1);
      en = lds_load(&ring.entry[k % ILU_RING]);
    }
    return __builtin_amdgcn_readfirstlane((uint32_t)en);
  };
  auto take = [&]() -> uint32_t {
    uint32_t q = 0;
    if (lane == 0) q = atomicAdd(&ring.head, 1u);
    q = __builtin_amdgcn_readfirstlane(q);
    const uint32_t k = q / B, j = q % B, r = k % ILU_RING;
    const uint32_t start = entry(k);
    if (lane == 0) atomicAdd(&ring.read[r], 1u);
    if (j == 0) {
      entry(k + 1);   /* drawn and back: k + 2 is drawn after it */
      put_k = k + 2;
      drawn = nrows;
      if (start < nrows && lane == 0) drawn = atomicAdd(ticket, B) - base;
    }
    return start + j;
  };
  auto put = [&]() {
    if (!put_k) return;
    const uint32_t r = put_k % ILU_RING;
    for (uint32_t n = 0; lds_load(&ring.read[r]) != B && n <= KF_SPIN_LIMIT; n++) __builtin_amdgcn_s_sleep(1);
    if (lane == 0) {
      lds_store(&ring.read[r], 0u);
      lds_store(&ring.entry[r], (unsigned long long)put_k << 32 | drawn);
    }
    put_k = 0;
  };

  /* a row's record, then its blocks, tables and L_old in one round of loads
   * (what lies beyond the round is loaded in load_rest) */
  uint32_t rv = 0, cv = 0, gv = 0, mo = 0, jv = 0;
  uint16_t ov = 0;
  T av[ILU_Q], lv[ILU_Q];
  ilu_row w;
  auto load_rec = [&](uint32_t t) { rv = t < nrows && lane < 6 ? rec[8 * (size_t)t + lane] : 0u; };
  auto load_row = [&]() {
    w.i = __builtin_amdgcn_readlane(rv, 0);
    w.j0 = __builtin_amdgcn_readlane(rv, 1);
    w.L = __builtin_amdgcn_readlane(rv, 2);
    w.nlow = __builtin_amdgcn_readlane(rv, 3);
    w.mbeg = __builtin_amdgcn_readlane(rv, 4);
    w.mcnt = __builtin_amdgcn_readlane(rv, 5);
    if (lane < w.nlow) {
      gv = ldiag[w.j0 + lane];
      mo = moff[w.j0 + lane];
      if (EXACT) cv = d.col[w.j0 + lane];
    } else {
      mo = w.mcnt;
    }
    if (lane < w.mcnt) { jv = mjm[w.mbeg + lane]; ov = mlo[w.mbeg + lane]; }
#pragma unroll
    for (int q = 0; q < ILU_Q; q++) {
      const uint32_t k = lane + 64 * q;
      if (k < 16 * w.L) av[q] = a[16 * (size_t)w.j0 + k];
      if (EXACT && k < 16 * w.nlow) {
        const uint32_t pp = k >> 4, ee = k & 15;
        lv[q] = pp == 0 ? a[16 * ((size_t)w.j0 + w.nlow - 1) + ee] : lold[16 * ((size_t)w.j0 + pp) + ee];
      }
    }
  };

  uint32_t t = take();
  load_rec(t);
  put();
  load_row();
  while (t < nrows) {
    const uint32_t i = w.i, j0 = w.j0, L = w.L, nlow = w.nlow, mcnt = w.mcnt, pd = w.nlow, moreg = mo;
    /* staged blocks: [0, nlow) inv(U(m,m)); EXACT: [nlow, 2 nlow) U(m,m);
     * from mbase the U(m,k) of the update pairs; from lbase (EXACT) L_old.
     * ssrc: where the published ones stand, in blocks of apub (the U(m,m)
     * follow its nnzb blocks). */
    const uint32_t mbase = EXACT ? 2 * nlow : nlow, nsrc = mbase + mcnt, lbase = nsrc + 8;
    for (uint32_t k = lane, first = 1; k < nlow; k += 64, first = 0) {
      ssrc[k] = first ? gv : ldiag[j0 + k];
      smoff[k] = first ? mo : moff[j0 + k];
      if (EXACT) ssrc[nlow + k] = nnzb + (first ? cv : d.col[j0 + k]);
    }
    for (uint32_t k = lane, first = 1; k < mcnt; k += 64, first = 0) {
      ssrc[mbase + k] = first ? jv : mjm[w.mbeg + k];
      slo[k] = 16 * (first ? ov : mlo[w.mbeg + k]);
    }
    if (lane < 8) slo[mcnt + lane] = 0;
    if (lane == 0) smoff[nlow] = mcnt;
    wave_lds_sync();
    /* the published blocks, QB values per lane per round (a lane past the
     * end reads the last block and drops it); a value still holding the
     * sentinel is loaded again.  While the first round is on its way the
     * row's own blocks go to LDS. */
    const uint32_t tot = 16 * nsrc;
    for (uint32_t b0 = 0; b0 == 0 || b0 < tot; b0 += 64 * QB) {
      uint32_t need = 0, blk[QB];
      T v[QB];
      if (tot) {
#pragma unroll
        for (int q = 0; q < QB; q++) blk[q] = ssrc[min(b0 / 16 + grp + 4 * q, nsrc - 1)];
#pragma unroll
        for (int q = 0; q < QB; q++) {
          v[q] = ld_coherent(apub + 16 * (size_t)blk[q] + e);
          if (b0 + lane + 64 * q < tot) need |= 1u << q;
        }
      }
      if (b0 == 0) {
#pragma unroll
        for (int q = 0; q < ILU_Q; q++) {
          const uint32_t k = lane + 64 * q;
          if (k < 16 * L) {
            sa[k] = av[q];
            if (EXACT) sa0[k] = av[q];
          }
          if (EXACT && k < 16 * nlow) stage[16 * lbase + k] = lv[q];
        }
        for (uint32_t k = lane + 64 * ILU_Q; k < 16 * L; k += 64) {
          const T x = a[16 * (size_t)j0 + k];
          sa[k] = x;
          if (EXACT) sa0[k] = x;
        }
        if (EXACT) {
          for (uint32_t k = lane + 64 * ILU_Q; k < 16 * nlow; k += 64)
            stage[16 * lbase + k] = lold[16 * ((size_t)j0 + (k >> 4)) + (k & 15)];
          wave_lds_sync();
          /* I A(i,k) of the upper blocks (in place: a group's lanes read
           * the whole block before they store it) */
          for (uint32_t p = pd + grp; p < L; p += 4) {
            const T *a0 = sa0 + 16 * p;
            T dq = T(0);
#pragma unroll
            for (int k = 0; k < 4; k++) dq += (er == (uint32_t)k ? T(1) : T(0)) * a0[4 * k + ec];
            sa0[16 * p + e] = dq;
          }
        }
      }
      for (uint32_t n = 0;; n++) {
#pragma unroll
        for (int q = 0; q < QB; q++)
          if ((need & (1u << q)) && sentinel<T>::raw(v[q]) != snt) {
            stage[b0 + lane + 64 * q] = v[q];
            need &= ~(1u << q);
          }
        if (!need || aborted) break;
        if (n >= KF_SPIN_LIMIT) {
          atomicOr(d.err, KF_ERR_SPIN_LIMIT);
          aborted = true;
          break;
        }
        for (uint32_t z = 0; z < d.spin_sleep; z++) __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int q = 0; q < QB; q++)
          if (need & (1u << q)) v[q] = ld_coherent(apub + 16 * (size_t)blk[q] + e);
      }
    }
    aborted = __any(aborted);   /* a wave gives up at most once per launch */
    /* nothing is waited for from here to the row's end: take the next ticket */
    t = take();
    load_rec(t);
    wave_lds_sync();

    if (EXACT) {
      /* L_old(i,m) U(m,m) of all lower blocks, four at a time, into L_old's place */
      for (uint32_t p = grp; p < nlow; p += 4) {
        T *q = stage + 16 * (lbase + p);
        const T dq = blk_mul(q, stage + 16 * (nlow + p), er, ec);
        q[e] = dq;
      }
      wave_lds_sync();
    }
    /* The elimination.  The row's chain is a(i,m) -> L(i,m) -> the updates
     * of row i -> the next a(i,m): every group of 16 lanes forms L(i,m) by
     * itself (its quads hold the block's rows, so the product needs no
     * exchange through LDS), and all operands of a step are read at once,
     * without a branch: the pairs' bounds are scalars, their targets are
     * known one step ahead, and a lane past the step's pairs works on some
     * other pair (the table ends in 8 spare ones) and does not store. */
    {
      uint32_t i0 = 0, i1 = step_end(moreg, smoff, 1);
      uint32_t o0 = slo[grp], o1 = slo[grp + 4];
      for (uint32_t p = 0; p < nlow; p++) {
        const bool on0 = i0 + grp < i1, on1 = i0 + grp + 4 < i1, two = i1 - i0 > 4;
        T v = sa[16 * p + e], dq = T(0), bi[4], u0[4], u1[4];
        if (EXACT) dq = stage[16 * (lbase + p) + e];
        const T t0 = sa[o0 + e], t1 = sa[o1 + e];
        blk_col(stage + 16 * p, ec, bi);
        blk_col(stage + 16 * (mbase + i0 + grp), ec, u0);
        if (two) blk_col(stage + 16 * (mbase + i0 + grp + 4), ec, u1);
        const uint32_t i2 = step_end(moreg, smoff, p + 2 < nlow ? p + 2 : nlow);
        const uint32_t n0 = slo[i1 + grp], n1 = slo[i1 + grp + 4];
        if (EXACT) {
          /* a(i,m) = (a - L_old U(m,m)) + L_old U(m,m) */
          v = T(-1) * dq + v;
          v = T(1) * dq + v;
        }
        const T lw = row_mul(v, bi);   /* L(i,m) = a(i,m) inv(U(m,m)) */
        if (grp == 0) sa[16 * p + e] = lw;
        /* a(i,k) -= L(i,m) U(m,k) for the update pairs of m (distinct k) */
        const T s0 = t0 - row_mul(lw, u0);
        if (on0) sa[o0 + e] = s0;
        if (two) {
          const T s1 = t1 - row_mul(lw, u1);
          if (on1) sa[o1 + e] = s1;
          for (uint32_t x = i0 + 8; x < i1; x += 4) {
            const uint32_t o2 = slo[x + grp];
            T u2[4];
            blk_col(stage + 16 * (mbase + x + grp), ec, u2);
            const T s2 = sa[o2 + e] - row_mul(lw, u2);
            if (x + grp < i1) sa[o2 + e] = s2;
          }
        }
        wave_lds_sync();
        i0 = i1;
        i1 = i2;
        o0 = n0;
        o1 = n1;
      }
    }

    if (EXACT) {
      /* upper blocks: a = (a - I A(i,k)) + I A(i,k), A = the fill's block */
      for (uint32_t p = pd + grp; p < L; p += 4) {
        const T dq = sa0[16 * p + e];
        T v = sa[16 * p + e];
        v = T(-1) * dq + v;
        v = T(1) * dq + v;
        sa[16 * p + e] = v;
      }
      wave_lds_sync();
      if (lane < 16) st_coherent(apub + 16 * ((size_t)nnzb + i) + e, canon(sa[16 * pd + e]));
    }
    /* published copies of what later rows read, as soon as they are final:
     * U(i,k) before the diagonal's inverse, both before this row's own stores */
    for (uint32_t k = 16 + lane; k < 16 * (L - pd); k += 64)
      st_coherent(apub + 16 * ((size_t)j0 + pd) + k, canon(sa[16 * pd + k]));
    {
      const T *s = sa + 16 * pd;
      T f[18];
#pragma unroll
      for (int q = 0; q < 18; q++) f[q] = s[(cof[q / 6] >> (4 * (q % 6))) & 15u];
      const T s0 = s[0], s1 = s[1], s2 = s[2], s3 = s[3];
      T acc = f[0];
      if (neg & 1u) acc = -acc;
      acc = acc * f[1] * f[2];
#pragma unroll
      for (int tt = 1; tt < 6; tt++) {
        const T pr = f[3 * tt] * f[3 * tt + 1] * f[3 * tt + 2];
        acc = (neg & (1u << tt)) ? acc - pr : acc + pr;
      }
      const T d0 = lane_get(acc, 0), d4 = lane_get(acc, 4), d8 = lane_get(acc, 8), d12 = lane_get(acc, 12);
      T det = s0 * d0 + s1 * d4 + s2 * d8 + s3 * d12;
      det = T(1) / det;
      acc *= det;
      wave_lds_sync();
      if (lane < 16) {
        st_coherent(apub + 16 * ((size_t)j0 + pd) + e, canon(acc));
        if (!isfinite((double)acc)) atomicOr(d.err, KF_ERR_NONFINITE_PIVOT);
        sa[16 * pd + e] = acc;
      }
    }
    put();
    if (t < nrows) load_row();
    wave_lds_sync();
    /* the factors, a block row of 4 values per lane and store */
    for (uint32_t k = lane; k < 4 * L; k += 64) {
      T x[4];
      ilu_ld4(sa + 4 * k, x);
      ilu_st4(a + 16 * (size_t)j0 + 4 * k, x);
      if (EXACT && k < 4 * nlow) ilu_st4(lold + 16 * (size_t)j0 + 4 * k, x);
      TS y[4];
#pragma unroll
      for (int q = 0; q < 4; q++) ilu_cvt(x[q], y + q);
      if (sizeof(TS) == 2) ilu_st4(reinterpret_cast<TS *>(out.abf) + 16 * (size_t)j0 + 4 * k, y);
      if (out.val) {
        /* slot p of L, slot p - nlow - 1 of U, or the diagonal */
        const uint32_t p = k >> 2, u = p > nlow ? p - nlow - 1 : p;
        const size_t slot = (size_t)(i >> 4) * out.K + u + (p > nlow ? (size_t)out.nslice * out.K : 0);
        TS *o = static_cast<TS *>(out.val) + 16 * (i & 15u) + 4 * (k & 3u);
        o += 256 * (p == nlow ? 2 * (size_t)out.nslice * out.K + (i >> 4) : slot);
        if (p == nlow || u < out.K) ilu_st4(o, y);
      }
    }
    wave_lds_sync();
  }
}

/* the slots other rows read -- each row's blocks from the diagonal on, and
 * with nu the U(i,i) after the nnzb blocks -- preset to the call's sentinel:
 * 16 lanes per row, 16 bytes each (all of A's blocks were preset before,
 * nearly twice the bytes) */
template <typename T>
__global__ __launch_bounds__(256) void k_ilu_preset(uint32_t N, const uint32_t *__restrict__ rowptr,
                                                    const uint32_t *__restrict__ diag, uint32_t nnzb, bool nu,
                                                    T *__restrict__ apub, typename sentinel<T>::bits snt)
{
  const uint32_t i = blockIdx.x * 16u + (threadIdx.x >> 4), l = threadIdx.x & 15u;
  if (i >= N) return;
  constexpr uint32_t V = 16 / sizeof(T);   /* values per store */
  union { typename sentinel<T>::bits b[V]; uint4 q; } w;
#pragma unroll
  for (uint32_t k = 0; k < V; k++) w.b[k] = snt;
  const size_t j = 16 * (size_t)diag[i], n = 16 * (size_t)rowptr[i + 1] - j;
  for (size_t k = V * l; k < n; k += 16 * V) *reinterpret_cast<uint4 *>(apub + j + k) = w.q;
  if (nu && V * l < 16) *reinterpret_cast<uint4 *>(apub + 16 * ((size_t)nnzb + i) + V * l) = w.q;
}

static uint32_t persistent_waves(uint32_t work, uint32_t cap)
{
  return work < cap ? (work ? work : 1) : cap;
}

/* true: the planned kernel ran, and wrote what `out` asks for */
template <typename T, bool EXACT, typename TS>
static bool launch_ilu(kf_ctx *c, T *a, T *lold, T *ud, const ilu_out &out)
{
  /* the context's setting, else what fits the registers: 2048 waves in FP64
   * (221 VGPRs, two per SIMD; capped at three the exact sweep spills and
   * takes twice as long), and for the single-precision factors (127 VGPRs)
   * 4096 where the schedule has that many rows to a level, 3072 below, where
   * waves that wait for later levels only crowd the polls (2.65M vertices:
   * 5.3 -> 4.6 ms; 161K: 0.87 against 0.90 ms) */
  const bool wide = (uint64_t)c->d.N >= 3072ull * (c->nlev_l ? c->nlev_l : 1);
  const uint32_t nw =
      persistent_waves(c->d.N, c->ilu_waves ? c->ilu_waves : sizeof(T) == 8 ? 2048u : wide ? 4096u : 3072u);
  const ilu_layout lay(c->ilu_maxrow, c->ilu_maxlow, c->ilu_maxmatch, sizeof(T), EXACT);
  /* wavefronts per workgroup and rows per batch: as asked, within the LDS */
  uint32_t G = c->ilu_group;
  const size_t lds_cap = c->lds_max - sizeof(ilu_ring);
  while (G > 1 && G * (size_t)lay.bytes > lds_cap) G--;
  if (lay.bytes <= lds_cap) {
    const uint32_t nb = (nw + G - 1) / G;
    /* published copies (the blocks of A, then the U(i,i)), preset to this
     * call's sentinel */
    const size_t na = 16 * (c->nnzb + (EXACT ? (size_t)c->d.N : 0));
    if (c->ilu_napub < na) {
      KF_CHECK(hipStreamSynchronize(c->stream));
      if (c->ilu_apub) KF_CHECK(hipFree(c->ilu_apub));
      KF_CHECK(hipMalloc(&c->ilu_apub, na * sizeof(double)));
      c->ilu_napub = na;
    }
    const typename sentinel<T>::bits snt = sentinel<T>::of(++c->icall);
    T *apub = (T *)c->ilu_apub;
    hipLaunchKernelGGL(k_ilu_preset<T>, dim3(kf_blocks_for(c->d.N, 16)), dim3(256), 0, c->stream, c->d.N, c->d.rowptr,
                       c->d.diag, (uint32_t)c->nnzb, EXACT, apub, snt);
    KF_LAUNCH_CHECK();
    if (G * (size_t)lay.bytes > 64 * 1024)
      KF_CHECK(hipFuncSetAttribute((const void *)k_ilu_rows<T, EXACT, TS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(G * lay.bytes)));
    const int s = kf_prof_begin(c, KP_ILU);
    hipLaunchKernelGGL((k_ilu_rows<T, EXACT, TS>), dim3(nb), dim3(64 * G), G * lay.bytes, c->stream, c->d, c->ilu_rec,
                       c->d.N, c->ticket + 2, c->ticket_base[2], G, (uint32_t)c->nnzb, apub, snt, a, lold, c->ilu_ldiag,
                       c->ilu_moff, c->ilu_mjm, c->ilu_mlo, c->ilu_maxrow, c->ilu_maxlow, c->ilu_maxmatch, out);
    KF_LAUNCH_CHECK();
    kf_prof_end(c, s);
    c->ticket_base[2] += kf_ticket_advance_ring(c->d.N, nb, G);
    return true;
  } else {
    const uint32_t epoch = ++c->epoch;
    const int s = kf_prof_begin(c, KP_ILU);
    hipLaunchKernelGGL((k_ilu<T, EXACT>), dim3(nw), dim3(64), 0, c->stream, c->d, c->lrows, c->d.N, c->ticket + 2,
                       c->ticket_base[2], c->rdone, epoch, a, lold, ud);
    KF_LAUNCH_CHECK();
    kf_prof_end(c, s);
    c->ticket_base[2] += c->d.N + nw;
    return false;
  }
}

__global__ __launch_bounds__(256) void k_to_bf16(size_t n, const float *__restrict__ src, uint16_t *__restrict__ dst)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  /* round to nearest even */
  uint32_t u = __float_as_uint(src[i]);
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7FFFu + lsb;
  dst[i] = (uint16_t)(u >> 16);
}

void kf_launch_ilu(kf_ctx *c)
{
  if (c->maxrow > ILU_MAXROW) {
    fprintf(stderr, "kf: ILU supports at most %d blocks per row (mesh has %u)\n", ILU_MAXROW, c->maxrow);
    abort();
  }
  const size_t n = 16 * c->nnzb;
  if (c->opt.prec == KF_PREC_BF16 && !c->abf) KF_CHECK(hipMalloc((void **)&c->abf, n * sizeof(uint16_t)));
  ilu_out out = {c->abf, NULL, 0, 0};
  if (c->opt.jacobi_sweeps > 0) out.val = kf_jac_slices(c, &out.K, &out.nslice);
  bool wrote;
  if (c->opt.prec == KF_PREC_FP64) {
    if (c->opt.ilu_exact) {
      if (!c->lold) {
        KF_CHECK(hipMalloc((void **)&c->lold, n * sizeof(double)));
        KF_CHECK(hipMemset(c->lold, 0, n * sizeof(double)));
        KF_CHECK(hipMalloc((void **)&c->ud, 16 * (size_t)c->d.N * sizeof(double)));
      }
      wrote = launch_ilu<double, true, double>(c, c->a64, c->lold, c->ud, out);
    } else {
      wrote = launch_ilu<double, false, double>(c, c->a64, NULL, NULL, out);
    }
  } else if (c->opt.prec == KF_PREC_FP32) {
    wrote = launch_ilu<float, false, float>(c, c->a32, NULL, NULL, out);
  } else {
    wrote = launch_ilu<float, false, uint16_t>(c, c->a32, NULL, NULL, out);
    if (!wrote) {
      hipLaunchKernelGGL(k_to_bf16, dim3(kf_blocks_for(n, 256)), dim3(256), 0, c->stream, n, c->a32, c->abf);
      KF_LAUNCH_CHECK();
    }
  }
  c->jsl_fresh = wrote && out.val;   /* else the sweeps pack the copy when they need it */
}
