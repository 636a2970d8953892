// Device-side definitions shared by every kernel of the library: argument
// structs, the Boys function, dual numbers and quartet lookup.
//
// Work decomposition.  Screened shell pairs are sorted by class and, within a
// class, by descending Schwarz bound.  Each contracted pair expands into its
// primitive pairs ("pseudo pairs", stored contiguously per pair); a contracted
// quartet is the sum of its pseudo-pair quartets.  For a bra pair the
// admissible kets of a class form a prefix of its list (Schwarz-sorted,
// canonical j <= i within one class), so a work list is a running-count array
// over the bra pairs.  The K, gradient and quadrature kernels give a workgroup
// one bra pair and a run of its kets and sum a contracted quartet's primitives
// in registers; the array-form kernels (qx_pairm.h) find a thread's quartet by
// binary search.  The stored integrals use the same lists over pseudo pairs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define QX_BLOCK 128      // threads per block of the array-form kernels; default of the streaming ones
#define QX_BLOCK_MAX 256  // largest block of the streaming J/K and gradient kernels (a multiple of 64)
#define QX_TWO_PI_5_2 34.986836655249725  // 2 pi^(5/2)
#define QX_PI 3.14159265358979323846

// Boys table: F_m(T_g) for T_g = g / QX_BOYS_INV_H, g = 0..QX_BOYS_NPTS-1,
// m = 0..QX_BOYS_NM-1.  A seven-term Taylor expansion about the nearest grid
// point (|T - T_g| <= 1/64) gives F_M; lower orders follow by downward
// recursion.  Above QX_BOYS_TMAX: asymptotic F_0 and upward recursion.
#define QX_BOYS_TMAX 36.0
#define QX_BOYS_INV_H 32.0
#define QX_BOYS_NM 24
#define QX_BOYS_NPTS (36 * 32 + 2)
#define QX_BOYS_MMAX (QX_BOYS_NM - 7)

// largest Cartesian shell-pair block (f x f); sizes the Schwarz diagonal rows
#define QX_PAIR_STRIDE 100

enum QxEpi {
  QX_EPI_STORE = 0,    // out[store_base + comp * nquart + t] (single-primitive bases)
  QX_EPI_SCHWARZ = 2,  // diagonal (f1 f2|f1 f2) of pair P into out[P * stride + f1*nb + f2]
  QX_EPI_JK = 3,       // direct J', K' accumulation with the density
  QX_EPI_GRAD = 5,     // adjoint gradient: sum dERI * density pair products
  QX_EPI_PAIRM = 7     // integrals or derivative slices into the function-pair matrix (qx_pairm.h)
};

struct QxPairsDev {        // screened shell pairs in sorted order (SoA)
  const double* Ax; const double* Ay; const double* Az;      // centre of shell a
  const double* ABx; const double* ABy; const double* ABz;   // A - B
  const int* sa; const int* sb;                              // shell indices
  const int* bfa; const int* bfb;                            // first Cartesian function
  const int* atom_a; const int* atom_b;
  const int* pp_first; const int* pp_n;                      // pseudo-pair range
};

struct QxPrimPairsDev {    // pseudo pairs (one primitive pair each), SoA
  const int* pair;                                           // owning pair
  const double* p;                                           // alpha + beta
  const double* Px; const double* Py; const double* Pz;      // product centre
  const double* K;      // c_a c_b exp(-alpha beta |AB|^2 / p)
  const double* a2;     // 2 alpha
  const double* b2;     // 2 beta
};

struct QxWorkDev {         // one (bra class, ket class) quartet list
  int bra_off, nbra;         // bra pseudo-pair range
  int ket_off, nket;         // ket pseudo-pair range
  const long long* prefix;   // nbra+1 running quartet counts
  const int* kstart;         // per bra pseudo pair: first admissible ket (null = 0)
  long long nquart;
  long long store_base;      // element offset of this list in the store buffer
  int diag;                  // kets are the pseudo pairs of the bra's own pair
};

struct QxEpiDev {
  int epi;
  int nbf, natom;
  int coord;                 // PAIRM derivatives: -1 = every coordinate's slice, else one coordinate
  int slice0, nslice;        // PAIRM derivatives: the slices are coordinates [slice0, slice0 + nslice) (nslice 0: coord rule)
  double* out;
  const double* D;           // density, Cartesian nbf x nbf (JK, GRAD)
  double* J; double* K;      // unsymmetrised J', K' (JK)
  int krows;                 // JK: K' rows of a workgroup's bra pair in LDS
  int kcols;                 // JK: width of those LDS rows (widest fragment's function range; 0 = nbf)
  const int* frag_col0;      // JK: first function of each fragment's range (null: 0); with pair_frag
  double* grad;              // GRAD: grad_copies x 3N accumulators (copy = block index % grad_copies)
  int grad_copies;           // GRAD: copies of the 3N accumulators (0 or 1: one)
  int grad_wred;             // GRAD: sum the bra centres' terms across the wavefront before LDS
  int grad_win;              // GRAD: widest LDS atom window in doubles (0 or >= QX_GRAD_LDS: QX_GRAD_LDS)
  const double* tv;          // 3N geometry direction: seed of the directional-derivative kernels
  int skip_single;           // PAIRM integrals: leave out quartets with all four centres on one atom
  const int* frag_skip;      // JK: per fragment, nonzero = leave its quartets out (null: none)
  const int* pair_frag;      // fragment of each sorted shell pair (fragmented contexts)
};

struct QxArgs {
  QxPairsDev pr;
  QxPrimPairsDev pp;
  QxWorkDev w;
  QxEpiDev e;
  const double* boys;
};

struct QxPairM;
struct QxKList;
struct QxJList;

struct QxLaunch {
  int fp32;                  // 1: recursion in FP32 (K / gradient); 2: derivative along tv (derivative slices)
  hipStream_t stream;
  int block;                 // JK / GRAD: threads per block (multiple of 64, <= QX_BLOCK_MAX; 0 = QX_BLOCK)
  const QxPairM* pm;         // PAIRM: the pair matrix and the contracted quartet list
  const QxKList* kl;         // the contracted quartet list (all but the array-form kernels)
};

__host__ __device__ inline int qx_launch_block(const QxLaunch* L) { return L->block > 0 ? L->block : QX_BLOCK; }

template <int M>
__device__ __forceinline__ void qx_boys(double T, const double* __restrict__ tab, double (&F)[M + 1]) {
  static_assert(M <= QX_BOYS_MMAX, "Boys order beyond table");
  if (T < QX_BOYS_TMAX) {
    const int g = (int)(T * QX_BOYS_INV_H + 0.5);
    const double d = g * (1.0 / QX_BOYS_INV_H) - T;
    const double* r = tab + g * QX_BOYS_NM + M;
    double f = r[6] * (1.0 / 720.0);
    f = f * d + r[5] * (1.0 / 120.0);
    f = f * d + r[4] * (1.0 / 24.0);
    f = f * d + r[3] * (1.0 / 6.0);
    f = f * d + r[2] * 0.5;
    f = f * d + r[1];
    f = f * d + r[0];
    F[M] = f;
    if constexpr (M > 0) {
      const double e = exp(-T);
      const double t2 = 2.0 * T;
#pragma unroll
      for (int m = M - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0 / (2 * m + 1));
    }
  } else {
    F[0] = 0.5 * sqrt(QX_PI / T);
    if constexpr (M > 0) {
      const double e = exp(-T);
      const double o2t = 0.5 / T;
#pragma unroll
      for (int m = 0; m < M; ++m) F[m + 1] = ((2 * m + 1) * F[m] - e) * o2t;
    }
  }
}

// ---- forward-mode (tangent) arithmetic --------------------------------
// A value and its derivative along one geometry direction tv (3N).  Tangent
// kernels run the generated recurrences in this type: the derivative part of
// a first-derivative integral is then a second derivative, contracted with
// tv on one index.
struct qx_dual {
  double v, d;
  __device__ __forceinline__ qx_dual() = default;
  __device__ __forceinline__ constexpr qx_dual(double x) : v(x), d(0.0) {}
  __device__ __forceinline__ constexpr qx_dual(double x, double y) : v(x), d(y) {}
};
__device__ __forceinline__ qx_dual operator+(qx_dual a, qx_dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ qx_dual operator-(qx_dual a, qx_dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ qx_dual operator-(qx_dual a) { return {-a.v, -a.d}; }
__device__ __forceinline__ qx_dual operator*(qx_dual a, qx_dual b) { return {a.v * b.v, a.v * b.d + a.d * b.v}; }
__device__ __forceinline__ qx_dual operator*(double a, qx_dual b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ qx_dual operator*(qx_dual a, double b) { return {a.v * b, a.d * b}; }
__device__ __forceinline__ qx_dual operator+(double a, qx_dual b) { return {a + b.v, b.d}; }
__device__ __forceinline__ qx_dual operator+(qx_dual a, double b) { return {a.v + b, a.d}; }
__device__ __forceinline__ qx_dual operator-(qx_dual a, double b) { return {a.v - b, a.d}; }
__device__ __forceinline__ qx_dual operator-(double a, qx_dual b) { return {a - b.v, -b.d}; }
__device__ __forceinline__ qx_dual operator/(qx_dual a, double b) { return {a.v / b, a.d / b}; }
__device__ __forceinline__ qx_dual& operator+=(qx_dual& a, qx_dual b) { a = a + b; return a; }
__device__ __forceinline__ qx_dual& operator-=(qx_dual& a, qx_dual b) { a = a - b; return a; }
__device__ __forceinline__ qx_dual& operator*=(qx_dual& a, qx_dual b) { a = a * b; return a; }

// F_m(T) along the tangent: dF_m/dT = -F_{m+1}
template <int M>
__device__ __forceinline__ void qx_boys_tan(qx_dual T, const double* __restrict__ tab, qx_dual (&F)[M + 1]) {
  double f[M + 2];
  qx_boys<M + 1>(T.v, tab, f);
#pragma unroll
  for (int m = 0; m <= M; ++m) F[m] = qx_dual(f[m], -T.d * f[m + 1]);
}

// Pair data of pseudo pair u (shell pair P) with its derivative along tv:
// centres move with their atoms, P = (alpha A + beta B) / p,
// K = c_a c_b exp(-alpha beta / p |A - B|^2).
struct QxTanPair {
  qx_dual K, P[3], A[3], AB[3];
};
__device__ __forceinline__ QxTanPair qx_tan_pair(const QxArgs& A_, int P, int u) {
  const double* tv = A_.e.tv;
  const int ta = 3 * A_.pr.atom_a[P], tb = 3 * A_.pr.atom_b[P];
  const double p = A_.pp.p[u], al = 0.5 * A_.pp.a2[u], be = 0.5 * A_.pp.b2[u];
  const double ab[3] = {A_.pr.ABx[P], A_.pr.ABy[P], A_.pr.ABz[P]};
  const double pv[3] = {A_.pp.Px[u], A_.pp.Py[u], A_.pp.Pz[u]};
  const double av[3] = {A_.pr.Ax[P], A_.pr.Ay[P], A_.pr.Az[P]};
  QxTanPair r;
  double abd = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const double dA = tv[ta + x], dB = tv[tb + x];
    r.A[x] = qx_dual(av[x], dA);
    r.AB[x] = qx_dual(ab[x], dA - dB);
    r.P[x] = qx_dual(pv[x], (al * dA + be * dB) / p);
    abd += ab[x] * (dA - dB);
  }
  const double K = A_.pp.K[u];
  r.K = qx_dual(K, -2.0 * al * be / p * abd * K);
  return r;
}

// Quartet t of the list: bra / ket pseudo pairs u1 / u2 and their pairs.
__device__ __forceinline__ void qx_locate(const QxArgs& A_, long long t, int& u1, int& u2, int& P1, int& P2) {
  const long long* pre = A_.w.prefix;
  int lo = 0, hi = A_.w.nbra;  // pre[lo] <= t < pre[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (pre[mid] <= t) lo = mid; else hi = mid;
  }
  const int local = (int)(t - pre[lo]);
  u1 = A_.w.bra_off + lo;
  P1 = A_.pp.pair[u1];
  u2 = A_.w.diag ? A_.pr.pp_first[P1] + local : A_.w.ket_off + (A_.w.kstart ? A_.w.kstart[lo] : 0) + local;
  P2 = A_.pp.pair[u2];
}

__device__ __forceinline__ void qx_atomic_add(double* p, double v) { unsafeAtomicAdd(p, v); }

__device__ __forceinline__ double qx_wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Degeneracy weight of a canonical quartet: 1/2 for each of a==b, c==d and
// (ab)==(cd), so that summing all 8 index permutations with this weight
// counts every distinct permutation once.
__device__ __forceinline__ double qx_degeneracy(const QxArgs& A_, int P1, int P2) {
  double f = 1.0;
  if (A_.pr.sa[P1] == A_.pr.sb[P1]) f *= 0.5;
  if (A_.pr.sa[P2] == A_.pr.sb[P2]) f *= 0.5;
  if (P1 == P2) f *= 0.5;
  return f;
}

// ---- ERI epilogues ----------------------------------------------------
template <int NA, int NB, int NC, int ND, typename R>
__device__ __forceinline__ void qx_epi_eri(const QxArgs& A_, long long t, int P1, int P2,
                                           const R (&o)[NA * NB * NC * ND], bool active) {
  constexpr int N = NA * NB * NC * ND;
  const int epi = A_.e.epi;
  if (!active) return;
  if (epi == QX_EPI_STORE) {
    double* out = A_.e.out + A_.w.store_base + t;
    const long long nq = A_.w.nquart;
#pragma unroll
    for (int k = 0; k < N; ++k) out[k * nq] = (double)o[k];
  } else if (epi == QX_EPI_SCHWARZ) {
    double* out = A_.e.out + (size_t)P1 * QX_PAIR_STRIDE;
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) qx_atomic_add(&out[i * NB + j], (double)o[((i * NB + j) * NC + i) * ND + j]);
  }
}

// ---- derivatives -------------------------------------------------------
__device__ __forceinline__ bool qx_single_atom(const QxArgs& A_, int P1, int P2) {
  const int a = A_.pr.atom_a[P1];
  return a == A_.pr.atom_b[P1] && a == A_.pr.atom_a[P2] && a == A_.pr.atom_b[P2];
}

// Output slice of nuclear coordinate y in a derivative-tensor pass (-1: not
// wanted): its place in the pass's range, or every slice (coord < 0), or only
// coordinate `coord` into slice 0.
__device__ __forceinline__ long long qx_dfull_slice(const QxEpiDev& e, int y) {
  if (e.nslice) return y >= e.slice0 && y < e.slice0 + e.nslice ? y - e.slice0 : -1;
  if (e.coord >= 0) return y == e.coord ? 0 : -1;
  return y;
}

// ---- kernel tables --------------------------------------------------------
#define QX_GRAD_LDS 768  // block-level gradient accumulators (3 x the atoms of a block's window)

#define QX_DPARTS_CAP 128  // most derivative parts one class may be split into
#define QX_JKPARTS_CAP 8  // most J/K parts (ranges of a components) of one class

struct QxClassEntry {
  int la, lb, lc, ld;
  int (*eri)(const QxArgs*, const QxLaunch*);      // integrals (store, Schwarz, pair matrix): array form or quadrature
  int (*deri)(const QxArgs*, const QxLaunch*);     // derivative (fp32 = 2: tangent) slices of the pair matrix
  int (*jkv)(const QxArgs*, const QxLaunch*);      // K of the directional derivative
  int (*hess)(const QxArgs*, const QxLaunch*);     // adjoint gradient's directional derivative
  int njk;
  int (*jk[QX_JKPARTS_CAP])(const QxArgs*, const QxLaunch*);  // K, per part
  double jk_flops[QX_JKPARTS_CAP];   // FP operations per primitive quartet, K epilogue included
  int nparts;
  int ngroups;
  int (*grad[QX_DPARTS_CAP])(const QxArgs*, const QxLaunch*);  // adjoint gradient, per part group
  double eri_flops;                   // algorithmic FP operations of one ERI body (J/K epilogue excluded)
  double part_flops[QX_DPARTS_CAP];   // same per derivative part, with the adjoint epilogue
  int part_ncomb[QX_DPARTS_CAP];      // derivative blocks (centre x direction) per part
  double group_flops[QX_DPARTS_CAP];  // sum of part_flops over each group
  int group_parts[QX_DPARTS_CAP];     // parts per group
};
