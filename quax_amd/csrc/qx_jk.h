// Integral-direct J and K.
//
// J and K are built by separate kernels, because J needs no (ab|cd) at all:
//   * J (qx_jeng_*): the density is expanded in Hermite Gaussians per primitive
//     pair, H_t = sum_ab E^ab_t D_ab, the Coulomb potential of all kets is
//     summed at every bra pair in the same basis,
//       P_t = sum_kets sum_tau (-1)^|tau| H_tau R_{t+tau},
//     and J_ab = sum_t E^ab_t P_t (McMurchie & Davidson 1978; Ahmadi & Almlof
//     1995).  A workgroup owns one bra primitive pair and walks all its kets,
//     so P_t stays in registers and J needs no atomics per quartet.  It
//     visits each pair of pairs twice (once as bra, once as ket).
//   * K (qx_kk_*): one workgroup owns one bra pair and a run of its kets.  K'
//     rows of the bra's functions, and the density rows that the contraction
//     reads, are in LDS for the whole run.
// A quartet's integrals are contracted over its primitives before the
// horizontal recurrence, so a contracted quartet updates K once.
//
// J is bound by instruction issue and the latency of its chains together (VALU
// issue 39-53 % of the cycles, FP64 24-32 %, for all bras below dd; 0.69 ms of
// 3.05 ms in all).  K of the light classes is bound by LDS atomics and the rows'
// flush (LDS busy 20-43 %), K of the d classes that stay here by their registers
// and scratch ((dp|pp), (dp|ds), (dd|ds): 0.5-2.2 KB per lane, 0.5-1.2 GB of HBM
// traffic per launch).  With J and K in one kernel, six streams of
// atomics per integral, the same pass took 8.5 ms.
#pragma once
#include "qx_device.h"

// One class's canonical quartet list over contracted pairs.
struct QxKList {
  int bra0, ket0;             // first sorted pair of the bra / ket class
  const long long* prefix;    // running quartet counts over the bra pairs
  const int* kstart;          // first admissible ket of each bra pair (null = 0)
  const int* n64;             // kets of each bra pair above the FP32 threshold (mixed precision)
  int sel;                    // 0: every ket; 1: the FP64 kets; 2: the FP32 kets
  int nbra;
  int maxket;                 // most kets of one bra pair
  long long nquart;
  int chunk;                  // kets per workgroup
  int ketprim;                // most primitives of a ket pair of the class
  int sub;                    // lanes that share one contracted quartet's primitives (one-lane kernels)
  int psplit;                 // workgroups that share them (quadrature kernels; grid z)
  const double* rys;          // Rys root and weight tables
  const int* frag_atoms;      // gradient: first atom and atom count of each fragment (null: one fragment)
};

struct QxRange {
  int first, count;
};

// Hermite density and potential of the J kernels, [t][pseudo pair of the class].
struct QxJList {
  int X;                      // bra pair class
  int npairs;
  int uoff[7];                // first pseudo pair of each class (and the end)
  int hoff[6];                // first element of each class's block
  const QxRange* range;       // [Y * npairs + pair]: the bra pair's admissible pseudo kets of class Y
  const int* n64;             // how many of them run in FP64 (mixed precision)
  unsigned f32_classes;       // mixed: bit Y set = the FP32 kernel takes the kets beyond n64, else FP64 takes all
  const double* H; double* P; // values
  const double* Hd; double* Pd;  // derivative parts (directional-derivative pass)
};

// K' rows and density rows of a workgroup in LDS: at most this much in all
// (one workgroup per CU still runs; two workgroups fit below half of it).
#define QX_K_LDS_MAX (160 * 1024)
// Density rows are staged only while two workgroups still share a CU: beyond,
// the occupancy they cost is worth more than the L2 reads they save.
#define QX_K_STAGE_MAX (80 * 1024)

__host__ __device__ constexpr int qx_ncart(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int qx_nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// What a pass accumulates: the value, or (directional derivative) its derivative.
__device__ __forceinline__ double qx_value(double x) { return x; }
__device__ __forceinline__ double qx_value(float x) { return (double)x; }
__device__ __forceinline__ double qx_value(qx_dual x) { return x.d; }

// ---- Hermite expansion coefficients --------------------------------------
// E[i][j][t] of one direction, i <= LA, j <= LB, t <= i + j (no prefactor).
template <int LA, int LB, typename R>
__device__ __forceinline__ void qx_herm_e(R PA, R PB, double o2p, R (&E)[LA + 1][LB + 1][LA + LB + 1]) {
#pragma unroll
  for (int i = 0; i <= LA; ++i)
#pragma unroll
    for (int j = 0; j <= LB; ++j)
#pragma unroll
      for (int t = 0; t <= LA + LB; ++t) {
        R v(0.0);
        if (i == 0 && j == 0) {
          if (t == 0) v = R(1.0);
        } else if (t <= i + j) {
          if (i > 0) {
            if (t > 0) v = v + o2p * E[i - 1][j][t - 1];
            if (t <= i - 1 + j) v = v + PA * E[i - 1][j][t];
            if (t + 1 <= i - 1 + j) v = v + (double)(t + 1) * E[i - 1][j][t + 1];
          } else {
            if (t > 0) v = v + o2p * E[i][j - 1][t - 1];
            if (t <= i + j - 1) v = v + PB * E[i][j - 1][t];
            if (t + 1 <= i + j - 1) v = v + (double)(t + 1) * E[i][j - 1][t + 1];
          }
        }
        E[i][j][t] = v;
      }
}

// Component k of angular momentum l in direction d (xx, xy, xz, yy, yz, zz).
__host__ __device__ constexpr int qx_comp(int l, int k, int d) {
  for (int i = 0, c = 0; i <= l; ++i)
    for (int j = 0; j <= i; ++j, ++c)
      if (c == k) return d == 0 ? l - i : d == 1 ? i - j : j;
  return 0;
}
// Exponent of Hermite index k in direction d, in the order t, u, v ascending
// over t + u + v <= L with v fastest.
__host__ __device__ constexpr int qx_herm(int L, int k, int d) {
  int c = 0;
  for (int t = 0; t <= L; ++t)
    for (int u = 0; u <= L - t; ++u)
      for (int v = 0; v <= L - t - u; ++v, ++c)
        if (c == k) return d == 0 ? t : d == 1 ? u : v;
  return 0;
}

// ---- density -> Hermite ---------------------------------------------------
template <typename R>
struct QxPairGeom {
  R K, PA[3], PB[3];
  double o2p;
};
__device__ __forceinline__ void qx_pair_geom(const QxArgs& A_, int P, int u, QxPairGeom<double>& g) {
  g.K = A_.pp.K[u];
  g.o2p = 0.5 / A_.pp.p[u];
  const double ab[3] = {A_.pr.ABx[P], A_.pr.ABy[P], A_.pr.ABz[P]};
  g.PA[0] = A_.pp.Px[u] - A_.pr.Ax[P];
  g.PA[1] = A_.pp.Py[u] - A_.pr.Ay[P];
  g.PA[2] = A_.pp.Pz[u] - A_.pr.Az[P];
#pragma unroll
  for (int d = 0; d < 3; ++d) g.PB[d] = g.PA[d] + ab[d];
}
__device__ __forceinline__ void qx_pair_geom(const QxArgs& A_, int P, int u, QxPairGeom<qx_dual>& g) {
  const QxTanPair t = qx_tan_pair(A_, P, u);
  g.K = t.K;
  g.o2p = 0.5 / A_.pp.p[u];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g.PA[d] = t.P[d] - t.A[d];
    g.PB[d] = g.PA[d] + t.AB[d];
  }
}
__device__ __forceinline__ void qx_split(double x, double* v, double*, long long k) { v[k] = x; }
__device__ __forceinline__ void qx_split(qx_dual x, double* v, double* d, long long k) { v[k] = x.v; d[k] = x.d; }
__device__ __forceinline__ void qx_join(const double* v, const double*, long long k, double& x) { x = v[k]; }
__device__ __forceinline__ void qx_join(const double* v, const double* d, long long k, qx_dual& x) { x = qx_dual(v[k], d[k]); }

// (-1)^|t| H_t of pseudo pair u: the ket sign is folded in.  A pair of
// different shells stands for both orders.
template <int LA, int LB, typename R>
__device__ __forceinline__ void qx_hermite_density(const QxArgs& A_, const QxJList& jl, int X, int u, double* H, double* Hd) {
  constexpr int NA = qx_ncart(LA), NB = qx_ncart(LB), L = LA + LB, NH = qx_nherm(L);
  const int P = A_.pp.pair[u], n = A_.e.nbf;
  const double* D = A_.e.D;
  const int ia = A_.pr.bfa[P], ib = A_.pr.bfb[P];
  const bool diag = A_.pr.sa[P] == A_.pr.sb[P];
  QxPairGeom<R> g;
  qx_pair_geom(A_, P, u, g);
  R Ex[LA + 1][LB + 1][L + 1], Ey[LA + 1][LB + 1][L + 1], Ez[LA + 1][LB + 1][L + 1];
  qx_herm_e<LA, LB>(g.PA[0], g.PB[0], g.o2p, Ex);
  qx_herm_e<LA, LB>(g.PA[1], g.PB[1], g.o2p, Ey);
  qx_herm_e<LA, LB>(g.PA[2], g.PB[2], g.o2p, Ez);
  R h[NH];
#pragma unroll
  for (int t = 0; t < NH; ++t) h[t] = R(0.0);
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      double d = D[(size_t)(ia + i) * n + ib + j];
      if (!diag) d += D[(size_t)(ib + j) * n + ia + i];
      const R kd = d * g.K;
      const int ax = qx_comp(LA, i, 0), ay = qx_comp(LA, i, 1), az = qx_comp(LA, i, 2);
      const int bx = qx_comp(LB, j, 0), by = qx_comp(LB, j, 1), bz = qx_comp(LB, j, 2);
#pragma unroll
      for (int t = 0; t < NH; ++t) {
        const int tx = qx_herm(L, t, 0), ty = qx_herm(L, t, 1), tz = qx_herm(L, t, 2);
        if (tx <= ax + bx && ty <= ay + by && tz <= az + bz) h[t] = h[t] + kd * (Ex[ax][bx][tx] * Ey[ay][by][ty] * Ez[az][bz][tz]);
      }
    }
  const long long m = jl.uoff[X + 1] - jl.uoff[X];
#pragma unroll
  for (int t = 0; t < NH; ++t) {
    const int s = qx_herm(L, t, 0) + qx_herm(L, t, 1) + qx_herm(L, t, 2);
    qx_split(s % 2 ? -h[t] : h[t], H, Hd, jl.hoff[X] + t * m + (u - jl.uoff[X]));
  }
}

// J_ab of contracted pair P from the Hermite potential, both orders.
template <int LA, int LB, typename R>
__device__ __forceinline__ void qx_hermite_potential(const QxArgs& A_, const QxJList& jl, int X, int P, double* J) {
  constexpr int NA = qx_ncart(LA), NB = qx_ncart(LB), L = LA + LB, NH = qx_nherm(L);
  const int n = A_.e.nbf;
  const int ia = A_.pr.bfa[P], ib = A_.pr.bfb[P];
  const bool diag = A_.pr.sa[P] == A_.pr.sb[P];
  const long long m = jl.uoff[X + 1] - jl.uoff[X];
  double o[NA * NB] = {};
  for (int u = A_.pr.pp_first[P]; u < A_.pr.pp_first[P] + A_.pr.pp_n[P]; ++u) {
    QxPairGeom<R> g;
    qx_pair_geom(A_, P, u, g);
    R Ex[LA + 1][LB + 1][L + 1], Ey[LA + 1][LB + 1][L + 1], Ez[LA + 1][LB + 1][L + 1];
    qx_herm_e<LA, LB>(g.PA[0], g.PB[0], g.o2p, Ex);
    qx_herm_e<LA, LB>(g.PA[1], g.PB[1], g.o2p, Ey);
    qx_herm_e<LA, LB>(g.PA[2], g.PB[2], g.o2p, Ez);
    R h[NH];
#pragma unroll
    for (int t = 0; t < NH; ++t) qx_join(jl.P, jl.Pd, jl.hoff[X] + t * m + (u - jl.uoff[X]), h[t]);
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int ax = qx_comp(LA, i, 0), ay = qx_comp(LA, i, 1), az = qx_comp(LA, i, 2);
        const int bx = qx_comp(LB, j, 0), by = qx_comp(LB, j, 1), bz = qx_comp(LB, j, 2);
        R v(0.0);
#pragma unroll
        for (int t = 0; t < NH; ++t) {
          const int tx = qx_herm(L, t, 0), ty = qx_herm(L, t, 1), tz = qx_herm(L, t, 2);
          if (tx <= ax + bx && ty <= ay + by && tz <= az + bz) v = v + (Ex[ax][bx][tx] * Ey[ay][by][ty] * Ez[az][bz][tz]) * h[t];
        }
        o[i * NB + j] += qx_value(g.K * v);
      }
  }
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      J[(size_t)(ia + i) * n + ib + j] = o[i * NB + j];
      if (!diag) J[(size_t)(ib + j) * n + ia + i] = o[i * NB + j];
    }
}

// ---- J: Hermite potential of one bra pseudo pair ---------------------------
// Geometry of a pseudo pair for the J kernels.
template <typename R>
struct QxCentre {
  R x[3];
};
__device__ __forceinline__ void qx_centre(const QxArgs& A_, int u, QxCentre<double>& c) {
  c.x[0] = A_.pp.Px[u]; c.x[1] = A_.pp.Py[u]; c.x[2] = A_.pp.Pz[u];
}
__device__ __forceinline__ void qx_centre(const QxArgs& A_, int u, QxCentre<qx_dual>& c) {
  const QxTanPair t = qx_tan_pair(A_, A_.pp.pair[u], u);
#pragma unroll
  for (int d = 0; d < 3; ++d) c.x[d] = t.P[d];
}
template <int M>
__device__ __forceinline__ void qx_boys_any(double T, const double* tab, double (&F)[M + 1]) { qx_boys<M>(T, tab, F); }
template <int M>
__device__ __forceinline__ void qx_boys_any(qx_dual T, const double* tab, qx_dual (&F)[M + 1]) { qx_boys_tan<M>(T, tab, F); }
__device__ __forceinline__ double qx_wave_total(double v) { return qx_wave_sum(v); }
__device__ __forceinline__ qx_dual qx_wave_total(qx_dual v) { return qx_dual(qx_wave_sum(v.v), qx_wave_sum(v.d)); }
__device__ __forceinline__ void qx_potential_add(double x, double* P, double*, long long k) { qx_atomic_add(&P[k], x); }
__device__ __forceinline__ void qx_potential_add(qx_dual x, double* P, double* Pd, long long k) {
  qx_atomic_add(&P[k], x.v);
  qx_atomic_add(&Pd[k], x.d);
}

// Adds the kets [v0, v1) of class Y (Hermite order L2) to the lane's j.  G:
// geometry and contraction (double or qx_dual); R: the R_tuv recursion's type
// (float in the FP32 part of a mixed pass).
template <int L1, int L2, typename G, typename R, class Core>
__device__ __forceinline__ void qx_j_kets(const QxArgs& A_, const QxJList& jl, int Y, int v0, int v1, double p,
                                          const QxCentre<G>& Pc, G (&j)[qx_nherm(L1)], Core core) {
  constexpr int L = L1 + L2, N2 = qx_nherm(L2);
  const long long m = jl.uoff[Y + 1] - jl.uoff[Y];
  for (int v = v0 + (int)threadIdx.x; v < v1; v += (int)blockDim.x) {
    const double q = A_.pp.p[v];
    QxCentre<G> Qc;
    qx_centre(A_, v, Qc);
    G h[N2];
#pragma unroll
    for (int t = 0; t < N2; ++t) qx_join(jl.H, jl.Hd, jl.hoff[Y] + t * m + (v - jl.uoff[Y]), h[t]);
    const double pq = p + q, al = p * q / pq;
    const G x = Pc.x[0] - Qc.x[0], y = Pc.x[1] - Qc.x[1], z = Pc.x[2] - Qc.x[2];
    G F[L + 1];
    qx_boys_any<L>(al * (x * x + y * y + z * z), A_.boys, F);
    double f = QX_TWO_PI_5_2 / (p * q * sqrt(pq));
    R b[L + 1];
#pragma unroll
    for (int k = 0; k <= L; ++k) {
      b[k] = R(f * F[k]);
      f *= -2.0 * al;
    }
    core(R(x), R(y), R(z), b, h, j);
  }
}

// J kernel of bra pairs of angular momentum L1: workgroup x = a bra pseudo
// pair of class jl.X, y = its share of every ket class.  FP32 (R = float):
// the kets beyond n64 of the classes in f32_classes, which the FP64 kernel of
// a mixed pass then leaves out.
#define QX_J_CASE(L1, L2)                                                                         \
  case L2:                                                                                        \
    qx_j_kets<L1, L2, G, R>(A_, jl, Y, v0, v1, p, Pc, j,                                           \
                            [](R x, R y, R z, const R (&b)[L1 + L2 + 1], const G (&h)[qx_nherm(L2)], \
                               G (&jj)[qx_nherm(L1)]) { qx_jc_##L1##L2<G, R>(x, y, z, b, h, jj); }); \
    break;
// (The kernels take the body as a macro: through a device function, the
// compiler kept a copy of the list argument in scratch, and the dual-number
// kernel of dd bras, 3.5 KB of scratch, then returned wrong potentials.  The
// build compares the kernels' scratch with what they need without a copy.)
#define QX_J_BODY(L1, bx, by, ny, ...)\
    const int u = jl.uoff[jl.X] + (int)(bx);                                                             \
    const int P = A_.pp.pair[u];                                                                  \
    if (A_.e.frag_skip && A_.e.frag_skip[A_.e.pair_frag[P]]) return;                              \
    constexpr int N1 = qx_nherm(L1);                                                              \
    constexpr bool F32 = sizeof(R) == 4;                                                          \
    G j[N1];                                                                                      \
    _Pragma("unroll") for (int t = 0; t < N1; ++t) j[t] = G(0.0);                                 \
    const double p = A_.pp.p[u];                                                                  \
    QxCentre<G> Pc;                                                                               \
    qx_centre(A_, u, Pc);                                                                         \
    for (int Y = 0; Y < 6; ++Y) {                                                                 \
      const QxRange r = jl.range[(size_t)Y * jl.npairs + P];                                      \
      int lo = 0, hi = r.count;                                                                   \
      if ((jl.f32_classes >> Y) & 1u) {                                                           \
        const int n64 = jl.n64[(size_t)Y * jl.npairs + P];                                        \
        if (F32) lo = n64; else hi = n64;                                                         \
      } else if (F32) {                                                                           \
        hi = 0;                                                                                   \
      }                                                                                           \
      const int len = hi - lo;                                                                    \
      if (len <= 0) continue;                                                                     \
      const int v0 = r.first + lo + (int)((long long)len * (by) / (ny));                              \
      const int v1 = r.first + lo + (int)((long long)len * ((by) + 1) / (ny));                        \
      switch (Y == 0 ? 0 : Y == 1 ? 1 : Y <= 3 ? 2 : Y - 1) {                                     \
        __VA_ARGS__                                                                               \
      }                                                                                           \
    }                                                                                             \
    const long long m = jl.uoff[jl.X + 1] - jl.uoff[jl.X];                                        \
    _Pragma("unroll") for (int t = 0; t < N1; ++t) {                                              \
      const G s = qx_wave_total(j[t]);                                                            \
      if (__lane_id() == 0) qx_potential_add(s, jl.P, jl.Pd, jl.hoff[jl.X] + t * m + (bx));         \
    }
#define QX_DEFINE_J_KERNEL(L1, WITH32, ...)                                                       \
  template <typename G, typename R>                                                               \
  __global__ __launch_bounds__(QX_BLOCK_MAX) void qx_jeng_##L1(QxArgs A_, QxJList jl) {           \
    QX_J_BODY(L1, blockIdx.x, blockIdx.y, gridDim.y, __VA_ARGS__)                                 \
  }                                                                                               \
  extern "C" int qx_launch_jengv_##L1(const QxArgs*, const QxJList*, int, int, hipStream_t);      \
  /* type: 0 FP64, 1 FP32 recursion, 2 derivative along tv */                                       \
  extern "C" int qx_launch_jeng_##L1(const QxArgs* a, const QxJList* jl, int type, int block, int split, hipStream_t s) { \
    const int nu = jl->uoff[jl->X + 1] - jl->uoff[jl->X];                                         \
    if (nu <= 0) return 0;                                                                        \
    if (type == 2) return qx_launch_jengv_##L1(a, jl, block, split, s);                           \
    const dim3 grid((unsigned)nu, (unsigned)split);                                               \
    if (type == 0) hipLaunchKernelGGL((qx_jeng_##L1<double, double>), grid, dim3(block), 0, s, *a, *jl); \
    else {                                                                                        \
      if constexpr (WITH32) hipLaunchKernelGGL((qx_jeng_##L1<double, float>), grid, dim3(block), 0, s, *a, *jl); \
      else return -1;                                                                             \
    }                                                                                             \
    return (int)hipGetLastError();                                                                \
  }
#define QX_DEFINE_JV_KERNEL(L1, ...)                                                              \
  __global__ __launch_bounds__(QX_BLOCK_MAX) void qx_jengv_##L1(QxArgs A_, QxJList jl) {          \
    using G = qx_dual;                                                                            \
    using R = qx_dual;                                                                            \
    QX_J_BODY(L1, blockIdx.x, blockIdx.y, gridDim.y, __VA_ARGS__)                                 \
  }                                                                                               \
  extern "C" int qx_launch_jengv_##L1(const QxArgs* a, const QxJList* jl, int block, int split, hipStream_t s) { \
    const dim3 grid((unsigned)(jl->uoff[jl->X + 1] - jl->uoff[jl->X]), (unsigned)split);          \
    hipLaunchKernelGGL(qx_jengv_##L1, grid, dim3(block), 0, s, *a, *jl);                          \
    return (int)hipGetLastError();                                                                \
  }

// ---- K rows -----------------------------------------------------------------
template <int NR, int NC>
__device__ __forceinline__ void qx_load_block(const double* d, int stride, double (&o)[NR * NC]) {
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) o[r * NC + c] = d[(size_t)r * stride + c];
}

// K workgroup: bra pair blockIdx.x, its kets blockIdx.y * chunk onwards.
// ROWS: K' rows in LDS (else global atomics); STAGE: density rows in LDS too.
struct QxKBlock {
  int P1, j0, j1, kst, W, col0;
};
__device__ __forceinline__ bool qx_k_block(const QxArgs& A_, const QxKList& kl, int i, int part, QxKBlock& b) {
  b.P1 = kl.bra0 + i;
  int lo = 0, hi = (int)(kl.prefix[i + 1] - kl.prefix[i]);
  if (kl.sel == 1) hi = min(hi, kl.n64[i]);
  if (kl.sel == 2) lo = min(hi, kl.n64[i]);
  b.j0 = lo + part * kl.chunk;
  b.j1 = min(hi, b.j0 + kl.chunk);
  if (b.j0 >= hi) return false;
  if (A_.e.frag_skip && A_.e.frag_skip[A_.e.pair_frag[b.P1]]) return false;
  b.kst = kl.ket0 + (kl.kstart ? kl.kstart[i] : 0);
  b.W = A_.e.kcols > 0 ? A_.e.kcols : A_.e.nbf;
  b.col0 = A_.e.frag_col0 ? A_.e.frag_col0[A_.e.pair_frag[b.P1]] : 0;
  return true;
}

__device__ __forceinline__ bool qx_k_block(const QxArgs& A_, const QxKList& kl, QxKBlock& b) {
  return qx_k_block(A_, kl, blockIdx.x, blockIdx.y, b);
}

// Zeroes the K' rows (and fills the density rows behind them).
template <int NA, int NB, bool STAGE>
__device__ __forceinline__ void qx_k_rows_begin(const QxArgs& A_, const QxKBlock& b, double* sk) {
  const int n = A_.e.nbf, ia = A_.pr.bfa[b.P1], ib = A_.pr.bfb[b.P1], len = (NA + NB) * b.W;
  for (int k = threadIdx.x; k < len; k += blockDim.x) sk[k] = 0.0;
  if (STAGE) {
    for (int r = 0; r < NA + NB; ++r) {
      const double* src = A_.e.D + (size_t)(r < NA ? ia + r : ib + r - NA) * n + b.col0;
      const int w = min(b.W, n - b.col0);
      for (int k = threadIdx.x; k < b.W; k += blockDim.x) sk[len + r * b.W + k] = k < w ? src[k] : 0.0;
    }
  }
  __syncthreads();
}

template <int NA, int NB>
__device__ __forceinline__ void qx_k_rows_end(const QxArgs& A_, const QxKBlock& b, const double* sk) {
  __syncthreads();
  const int n = A_.e.nbf, ia = A_.pr.bfa[b.P1], ib = A_.pr.bfb[b.P1];
  for (int r = 0; r < NA + NB; ++r) {
    double* dst = A_.e.K + (size_t)(r < NA ? ia + r : ib + r - NA) * n + b.col0;
    for (int k = threadIdx.x; k < b.W; k += blockDim.x) {
      const double v = sk[r * b.W + k];
      if (v != 0.0) qx_atomic_add(&dst[k], v);
    }
  }
}

template <int NA, int NB, int NC, int ND, bool ROWS>
__device__ __forceinline__ void qx_k_add(const QxArgs& A_, const QxKBlock& b, int P2, double* sk,
                                         const double (&kac)[NA * NC], const double (&kad)[NA * ND],
                                         const double (&kbc)[NB * NC], const double (&kbd)[NB * ND]) {
  const double fk = 2.0 * qx_degeneracy(A_, b.P1, P2);
  const int n = A_.e.nbf;
  const int ic = A_.pr.bfa[P2], id = A_.pr.bfb[P2];
  double *ra, *rb;
  int w, cc, cd;
  if (ROWS) {
    ra = sk; rb = sk + NA * b.W; w = b.W; cc = ic - b.col0; cd = id - b.col0;
  } else {
    ra = A_.e.K + (size_t)A_.pr.bfa[b.P1] * n; rb = A_.e.K + (size_t)A_.pr.bfb[b.P1] * n; w = n; cc = ic; cd = id;
  }
  auto add = [&](double* p, double v) {
    if (ROWS) atomicAdd(p, v);
    else qx_atomic_add(p, v);
  };
#pragma unroll
  for (int k = 0; k < NA * NC; ++k) add(&ra[(k / NC) * w + cc + k % NC], fk * kac[k]);
#pragma unroll
  for (int k = 0; k < NA * ND; ++k) add(&ra[(k / ND) * w + cd + k % ND], fk * kad[k]);
#pragma unroll
  for (int k = 0; k < NB * NC; ++k) add(&rb[(k / NC) * w + cc + k % NC], fk * kbc[k]);
#pragma unroll
  for (int k = 0; k < NB * ND; ++k) add(&rb[(k / ND) * w + cd + k % ND], fk * kbd[k]);
}

// K kernel of a light class: one lane per contracted quartet.
#define QX_DEFINE_K_BODY(NAME, NA, NB, NC, ND)                                                    \
  template <typename R, bool ROWS, bool STAGE>                                                    \
  __device__ __forceinline__ void qx_kd_##NAME(const QxArgs& A_, const QxKList& kl, const QxKBlock& b, double* qx_sk) { \
    if (ROWS) qx_k_rows_begin<NA, NB, STAGE>(A_, b, qx_sk);                                       \
    const int n_ = A_.e.nbf;                                                                      \
    for (int t = (int)threadIdx.x; t < (b.j1 - b.j0) * kl.sub; t += (int)blockDim.x) {            \
      const int j = b.j0 + t / kl.sub, s = t % kl.sub;                                            \
      const int P2 = b.kst + j;                                                                   \
      const int ic = A_.pr.bfa[P2], id = A_.pr.bfb[P2];                                           \
      double Dac[NA * NC], Dad[NA * ND], Dbc[NB * NC], Dbd[NB * ND];                              \
      if (STAGE) {                                                                                \
        const double *da = qx_sk + (NA + NB) * b.W - b.col0, *db = da + NA * b.W;                 \
        qx_load_block<NA, NC>(da + ic, b.W, Dac);                                                 \
        qx_load_block<NA, ND>(da + id, b.W, Dad);                                                 \
        qx_load_block<NB, NC>(db + ic, b.W, Dbc);                                                 \
        qx_load_block<NB, ND>(db + id, b.W, Dbd);                                                 \
      } else {                                                                                    \
        const double *da = A_.e.D + (size_t)A_.pr.bfa[b.P1] * n_, *db = A_.e.D + (size_t)A_.pr.bfb[b.P1] * n_; \
        qx_load_block<NA, NC>(da + ic, n_, Dac);                                                  \
        qx_load_block<NA, ND>(da + id, n_, Dad);                                                  \
        qx_load_block<NB, NC>(db + ic, n_, Dbc);                                                  \
        qx_load_block<NB, ND>(db + id, n_, Dbd);                                                  \
      }                                                                                           \
      double kac[NA * NC] = {}, kad[NA * ND] = {}, kbc[NB * NC] = {}, kbd[NB * ND] = {};          \
      qx_kb_##NAME<R>(A_, b.P1, P2, s, kl.sub, Dac, Dad, Dbc, Dbd, kac, kad, kbc, kbd);           \
      qx_k_add<NA, NB, NC, ND, ROWS>(A_, b, P2, qx_sk, kac, kad, kbc, kbd);                       \
    }                                                                                             \
    if (ROWS) qx_k_rows_end<NA, NB>(A_, b, qx_sk);                                                \
  }
#define QX_DEFINE_KK(NAME, NA, NB, NC, ND)                                                        \
  QX_DEFINE_K_BODY(NAME, NA, NB, NC, ND)                                                          \
  template <typename R, bool ROWS, bool STAGE>                                                    \
  __global__ __launch_bounds__(QX_BLOCK_MAX) void qx_kk_##NAME(QxArgs A_, QxKList kl) {           \
    HIP_DYNAMIC_SHARED(double, qx_sk)                                                             \
    QxKBlock b;                                                                                   \
    if (qx_k_block(A_, kl, b)) qx_kd_##NAME<R, ROWS, STAGE>(A_, kl, b, qx_sk);                    \
  }                                                                                               \
  QX_DEFINE_K_GO(NAME, NA, NB)

// Launcher of a K kernel template <R, ROWS, STAGE>: K' rows in LDS when they
// fit, density rows too when both do.
#define QX_DEFINE_K_GO(NAME, NA, NB)                                                              \
  template <typename R>                                                                           \
  static int qx_k_go_##NAME(const QxArgs* a, const QxLaunch* L) {                                 \
    const QxKList& kl = *L->kl;                                                                   \
    const int bs = qx_launch_block(L);                                                            \
    if (bs % 64 || bs > QX_BLOCK_MAX) return (int)hipErrorInvalidValue;                           \
    const size_t W = a->e.kcols > 0 ? a->e.kcols : a->e.nbf, rows = ((NA) + (NB)) * W * sizeof(double); \
    const bool fit1 = a->e.krows && rows <= QX_K_LDS_MAX, fit2 = fit1 && 2 * rows <= QX_K_STAGE_MAX; \
    const dim3 grid((unsigned)kl.nbra, (unsigned)((kl.maxket + kl.chunk - 1) / kl.chunk));        \
    if (fit2) hipLaunchKernelGGL((qx_kk_##NAME<R, true, true>), grid, dim3(bs), 2 * rows, L->stream, *a, kl); \
    else if (fit1) hipLaunchKernelGGL((qx_kk_##NAME<R, true, false>), grid, dim3(bs), rows, L->stream, *a, kl); \
    else hipLaunchKernelGGL((qx_kk_##NAME<R, false, false>), grid, dim3(bs), 0, L->stream, *a, kl); \
    return (int)hipGetLastError();                                                                \
  }
// FP64 and FP32 K kernels of a class, and (KV) K of the directional derivative.
#define QX_DEFINE_K_KERNEL(NAME, NA, NB, NC, ND, WITH32)                                          \
  QX_DEFINE_KK(NAME, NA, NB, NC, ND)                                                              \
  extern "C" int qx_launchj_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    if (L->fp32) {                                                                                \
      if constexpr (WITH32) return qx_k_go_##NAME<float>(a, L);                                   \
      return -1;                                                                                  \
    }                                                                                             \
    return qx_k_go_##NAME<double>(a, L);                                                          \
  }
#define QX_DEFINE_KV_KERNEL(NAME, NA, NB, NC, ND)                                                 \
  QX_DEFINE_KK(v##NAME, NA, NB, NC, ND)                                                           \
  extern "C" int qx_launchv_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    return a->e.tv ? qx_k_go_v##NAME<qx_dual>(a, L) : -1;                                         \
  }

// ---- small s, p molecules ------------------------------------------------------
// Every K and J list of a context without d shells in one launch: the lists'
// workgroups one after the other, each of QX_SMALL_BLOCK threads.  A molecule
// of a few atoms leaves most of the device idle in any one of the nine
// kernels, whose times (7-16 us each, a chain of loads and one primitive loop)
// and launches then add up.
#define QX_SMALL_BLOCK 128
struct QxSmall {
  QxKList k[6];   // 0000, 1000, 1010, 1100, 1110, 1111
  QxJList j[3];   // bra ss, ps, pp
  int end[9];     // workgroups of the lists up to each one
  int split;      // workgroups that share a J bra's kets
};
// (One branch with bx, by formed once: three of them took 18 registers more and
// 4 %, J/K of 64 waters 151 -> 158 us.)
#define QX_SMALL_J(L1, ...)                                                                       \
  {                                                                                               \
    using G = double;                                                                             \
    using R = double;                                                                             \
    const QxJList& jl = sm.j[L1];                                                                 \
    QX_J_BODY(L1, bx, by, sm.split, __VA_ARGS__)                                                  \
  }
#define QX_DEFINE_SMALL()                                                                         \
  __global__ __launch_bounds__(QX_SMALL_BLOCK) void qx_small(QxArgs A_, QxSmall sm) {             \
    HIP_DYNAMIC_SHARED(double, qx_sk)                                                             \
    const int w = blockIdx.x;                                                                     \
    int i = 0;                                                                                    \
    while (i < 8 && w >= sm.end[i]) ++i;                                                          \
    const int at = w - (i ? sm.end[i - 1] : 0);                                                   \
    if (i >= 6) {                                                                                 \
      const int by = at % sm.split, bx = at / sm.split;                                           \
      if (i == 6) QX_SMALL_J(0, QX_SMALL_CASES_0)                                                 \
      else if (i == 7) QX_SMALL_J(1, QX_SMALL_CASES_1)                                            \
      else QX_SMALL_J(2, QX_SMALL_CASES_2)                                                        \
      return;                                                                                     \
    }                                                                                             \
    const QxKList& kl = sm.k[i];                                                                  \
    QxKBlock b;                                                                                   \
    if (!qx_k_block(A_, kl, at % kl.nbra, at / kl.nbra, b)) return;                               \
    switch (i) {                                                                                  \
      case 0: qx_kd_e0000_0<double, true, true>(A_, kl, b, qx_sk); break;                         \
      case 1: qx_kd_e1000_0<double, true, true>(A_, kl, b, qx_sk); break;                         \
      case 2: qx_kd_e1010_0<double, true, true>(A_, kl, b, qx_sk); break;                         \
      case 3: qx_kd_e1100_0<double, true, true>(A_, kl, b, qx_sk); break;                         \
      case 4: qx_kd_e1110_0<double, true, true>(A_, kl, b, qx_sk); break;                         \
      default: qx_kd_e1111_0<double, true, true>(A_, kl, b, qx_sk); break;                        \
    }                                                                                             \
  }                                                                                               \
  extern "C" int qx_launch_small(const QxArgs* a, const QxSmall* sm, unsigned lds, hipStream_t s) { \
    if (sm->end[8] <= 0) return 0;                                                                \
    hipLaunchKernelGGL(qx_small, dim3((unsigned)sm->end[8]), dim3(QX_SMALL_BLOCK), lds, s, *a, *sm); \
    return (int)hipGetLastError();                                                                \
  }
