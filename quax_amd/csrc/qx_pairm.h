// Pair-matrix form of the integral and derivative tensors.
//
// The (n, n, n, n) tensor holds every integral up to eight times.  Writing
// those eight places from the lane that computed it costs eight scattered
// 8-byte stores (atomic ones for derivatives and contracted shells), and the
// lanes of a wavefront hold kets sorted by Schwarz bound, so no two of them
// share a cache line.  Instead a quartet's block goes to a matrix M over
// Cartesian function pairs, M[row of (a, b)][column of (c, d)], whose index is
//   class base + component * (pairs of the class) + (pair position):
// consecutive lanes (consecutive ket pairs) write consecutive doubles, each
// element once, also for contracted shells, whose primitive quartets are summed
// before the store (derivatives of contracted quartets add up in M by atomics).
// A quarter of the tensor's bytes is written this way; the runtime then
// brings M to AO functions in a spherical basis (qxk_pairm_ao), mirrors it
// (qxk_pairm_sym) and expands it row by row into the tensor with coalesced
// stores (qxk_pairm_expand).
#pragma once
#include "qx_device.h"

struct QxPairM {
  double* M;                 // slice y starts at M + y * slice
  long long ld, slice;
  int row0, rown, rowp;      // bra class: first row, pairs, first sorted pair
  int col0, coln, colp;      // ket class
  const long long* prefix;   // running contracted-quartet counts over the bra pairs (nbra + 1)
  const int* kstart;         // per bra pair: first admissible ket pair (null = 0)
  int nbra;
  long long nquart;          // contracted quartets
  int sub;                   // adjacent lanes that share one contracted quartet's primitives (array-form kernels): a
                             // power of two up to 64
  long long t0;              // number of the first one (a panel of bra pairs starts inside the list)
};

// Contracted quartet t of the list: its bra and ket pairs.
__device__ __forceinline__ void qx_locate_pairs(const QxPairM& pm, long long t, int& P1, int& P2) {
  t += pm.t0;
  int lo = 0, hi = pm.nbra;  // prefix[lo] <= t < prefix[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (pm.prefix[mid] <= t) lo = mid; else hi = mid;
  }
  P1 = pm.rowp + lo;
  P2 = pm.colp + (pm.kstart ? pm.kstart[lo] : 0) + (int)(t - pm.prefix[lo]);
}

template <int NAB, int NCD, typename R>
__device__ __forceinline__ void qx_pairm_eri(const QxPairM& pm, int P1, int P2, bool lead, R (&o)[NAB * NCD]) {
  if (pm.sub > 1) {  // launch-uniform
#pragma unroll
    for (int k = 0; k < NAB * NCD; ++k)
      for (int off = pm.sub >> 1; off > 0; off >>= 1) o[k] += __shfl_xor(o[k], off);
  }
  if (!lead) return;
  double* m = pm.M + (long long)(pm.row0 + P1 - pm.rowp) * pm.ld + pm.col0 + (P2 - pm.colp);
#pragma unroll
  for (int ij = 0; ij < NAB; ++ij)
#pragma unroll
    for (int kl = 0; kl < NCD; ++kl) m[(long long)ij * pm.rown * pm.ld + (long long)kl * pm.coln] = (double)o[ij * NCD + kl];
}

// ---- array-form kernels ---------------------------------------------------
// The integral cores add to their output array, so that a PAIRM launch sums its
// primitive quartets in place: one lane per contracted quartet, or pm.sub of
// them in a small molecule, each a share, and the shares meet in cross-lane sums
// (by atomics, the tensor of 8 atoms in a minimal basis took 442 us against 138).
// The other epilogues run one lane per primitive quartet.
struct QxArrayQuartet {
  int P1, P2, u1, u2, n1, n2, k0, ks;  // primitive quartets k0, k0 + ks, ...
};
__device__ __forceinline__ bool qx_array_quartet(const QxArgs& A_, const QxPairM& pm, long long t, QxArrayQuartet& q) {
  if (A_.e.epi == QX_EPI_PAIRM) {
    if (t >= pm.nquart * pm.sub) return false;
    q.ks = pm.sub;
    q.k0 = (int)(t % pm.sub);
    qx_locate_pairs(pm, t / pm.sub, q.P1, q.P2);
    q.u1 = A_.pr.pp_first[q.P1];
    q.u2 = A_.pr.pp_first[q.P2];
    q.n1 = A_.pr.pp_n[q.P1];
    q.n2 = A_.pr.pp_n[q.P2];
  } else {
    if (t >= A_.w.nquart) return false;
    qx_locate(A_, t, q.u1, q.u2, q.P1, q.P2);
    q.n1 = q.n2 = q.ks = 1;
    q.k0 = 0;
  }
  return true;
}

static inline dim3 qx_array_grid(const QxArgs* a, const QxLaunch* L, long long& nq) {
  nq = a->e.epi == QX_EPI_PAIRM ? (L->pm ? L->pm->nquart * L->pm->sub : 0) : a->w.nquart;
  return dim3((unsigned)((nq + QX_BLOCK - 1) / QX_BLOCK));
}

// Array-form ERI kernel: pair-matrix / store / Schwarz epilogues.
#define QX_DEFINE_ERI_KERNEL(NAME, N, NA, NB, NC, ND)                                             \
  __global__ __launch_bounds__(QX_BLOCK) void qx_k_##NAME(QxArgs A_, QxPairM pm) {                \
    const long long t = (long long)blockIdx.x * QX_BLOCK + threadIdx.x;                          \
    QxArrayQuartet q{};                                                                           \
    bool on = qx_array_quartet(A_, pm, t, q);                                                     \
    if (on && A_.e.skip_single) on = !qx_single_atom(A_, q.P1, q.P2);                             \
    double o[N] = {};                                                                             \
    if (on)                                                                                       \
      for (int k = q.k0; k < q.n1 * q.n2; k += q.ks)                                              \
        qx_core_##NAME<double>(A_, q.P1, q.P2, q.u1 + k / q.n2, q.u2 + k % q.n2, o);              \
    /* every lane: the sums over a quartet's lanes are cross-lane */                              \
    if (A_.e.epi == QX_EPI_PAIRM) qx_pairm_eri<NA * NB, NC * ND, double>(pm, q.P1, q.P2, on && q.k0 == 0, o); \
    else qx_epi_eri<NA, NB, NC, ND, double>(A_, t, q.P1, q.P2, o, on);                            \
  }                                                                                               \
  extern "C" int qx_launch_##NAME(const QxArgs* a, const QxLaunch* L) {                           \
    long long nq;                                                                                 \
    const dim3 grid = qx_array_grid(a, L, nq);                                                    \
    if (nq <= 0) return 0;                                                                        \
    if (L->fp32 || a->e.epi == QX_EPI_JK) return -1;                                              \
    const QxPairM pm = L->pm ? *L->pm : QxPairM{};                                                \
    hipLaunchKernelGGL(qx_k_##NAME, grid, dim3(QX_BLOCK), 0, L->stream, *a, pm);                  \
    return (int)hipGetLastError();                                                                \
  }
