// One-electron integrals (overlap, kinetic, nuclear attraction) and their
// contracted first derivatives, one kernel pair per shell-pair class (la, lb)
// with la >= lb <= 2 and generated attraction recurrences.
//
// Attraction: eight lanes share a shell pair and take every eighth nucleus
// each.  A lane adds its [e|0] integrals over nuclei and primitives in
// registers (the transfer to (a|b) depends on neither), the eight partial
// sums meet in three cross-lane steps and one lane transfers and stores the
// block.  Overlap and kinetic energy come from 1D Obara-Saika tables, one lane
// per pair, in the blocks of grid row 1 (values) or rows 1..6, one per centre
// and direction (derivatives), so that neither waits for the attraction
// loops.  Work is O(pairs x nuclei) on registers; the earlier form, one lane
// per ordered pair with the nuclei in sequence and its tables in 5-10 KB of
// scratch, was bound by that scratch's latency (280 functions, S, T, V and
// their contracted gradient: 8.5 ms, now 0.13 ms in twelve launches).
#pragma once
#include "qx_runtime.h"

struct QxOei {
  QxShellsDev sh;
  const double* boys;
  const int* la; const int* lb;  // shells of the class's two angular momenta
  int nla, nlb, npair;           // npair: nla * nlb, or the triangle when they are one list
  double* S; double* T; double* V;
  const double* Pd; const double* Wd; double* grad;
  const double* tv;              // geometry direction (dual-number kernels)
};

#define QX_OEI_LANES 8   // lanes per pair in the attraction blocks
#define QX_OEI_BLOCK 128

// Shells of pair t.
__device__ __forceinline__ void oei_pair(const QxOei& A, int t, bool same, int& sa, int& sb) {
  int i, j;
  if (same) {
    i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((i + 1) * (i + 2) / 2 <= t) ++i;
    while (i * (i + 1) / 2 > t) --i;
    j = t - i * (i + 1) / 2;
  } else {
    i = t / A.nlb;
    j = t - i * A.nlb;
  }
  sa = A.la[i];
  sb = A.lb[j];
}

template <typename R>
struct OeiPos {
  R x[3];
};
__device__ __forceinline__ void oei_atom(const QxOei& A, int at, OeiPos<double>& r) {
#pragma unroll
  for (int d = 0; d < 3; ++d) r.x[d] = A.sh.xyz[3 * at + d];
}
__device__ __forceinline__ void oei_atom(const QxOei& A, int at, OeiPos<qx_dual>& r) {
#pragma unroll
  for (int d = 0; d < 3; ++d) r.x[d] = qx_dual(A.sh.xyz[3 * at + d], A.tv[3 * at + d]);
}
__device__ __forceinline__ double oei_exp(double x) { return exp(x); }
__device__ __forceinline__ qx_dual oei_exp(qx_dual x) {
  const double e = exp(x.v);
  return qx_dual(e, e * x.d);
}
__device__ __forceinline__ double oei_out(double x) { return x; }
__device__ __forceinline__ double oei_out(qx_dual x) { return x.d; }
template <int M>
__device__ __forceinline__ void oei_boys(double T, const double* tab, double (&F)[M + 1]) { qx_boys<M>(T, tab, F); }
template <int M>
__device__ __forceinline__ void oei_boys(qx_dual T, const double* tab, qx_dual (&F)[M + 1]) {
  qx_boys_tan<M>(T, tab, F);
}

// Primitive pair: exponents, product centre relative to A, prefactor.
template <typename R>
struct OeiPrim {
  double a, b, p, oo2p;
  R K, P[3], PA[3], PB[3];
};
template <typename R>
__device__ __forceinline__ OeiPrim<R> oei_prim(const QxOei& A, const OeiPos<R>& a, const OeiPos<R>& b, int ia, int ib) {
  OeiPrim<R> r;
  r.a = A.sh.exps[ia];
  r.b = A.sh.exps[ib];
  r.p = r.a + r.b;
  const double op = 1.0 / r.p;
  r.oo2p = 0.5 * op;
  R ab2(0.0);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r.P[d] = (r.a * a.x[d] + r.b * b.x[d]) * op;
    r.PA[d] = r.P[d] - a.x[d];
    r.PB[d] = r.P[d] - b.x[d];
    const R ab = a.x[d] - b.x[d];
    ab2 = ab2 + ab * ab;
  }
  r.K = A.sh.coefs[ia] * A.sh.coefs[ib] * oei_exp(-r.a * r.b * op * ab2);
  return r;
}

// 1D overlap tables s[d][i][j], i <= IM, j <= JM (no prefactor).
template <int IM, int JM, typename R>
__device__ __forceinline__ void oei_s1d(const OeiPrim<R>& P, R (&s)[3][IM + 1][JM + 1]) {
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int j = 0; j <= JM; ++j)
#pragma unroll
      for (int i = 0; i <= IM; ++i) {
        if (i == 0 && j == 0) { s[d][i][j] = R(1.0); continue; }
        R v(0.0);
        if (j == 0) {
          v = P.PA[d] * s[d][i - 1][0];
          if (i > 1) v = v + (P.oo2p * (i - 1)) * s[d][i - 2][0];
        } else {
          v = P.PB[d] * s[d][i][j - 1];
          if (i > 0) v = v + (P.oo2p * i) * s[d][i - 1][j - 1];
          if (j > 1) v = v + (P.oo2p * (j - 1)) * s[d][i][j - 2];
        }
        s[d][i][j] = v;
      }
}

// 1D kinetic factor of (i, j).
template <int IM, int JM, typename R>
__device__ __forceinline__ R oei_t1(const R (&s)[IM + 1][JM + 1], double b, int i, int j) {
  R t = (b * (2 * j + 1)) * s[i][j] - (2.0 * b * b) * s[i][j + 2];
  if (j > 1) t = t - (0.5 * j * (j - 1)) * s[i][j - 2];
  return t;
}

// component k of angular momentum l, in the order xx, xy, xz, yy, yz, zz
__host__ __device__ constexpr int oei_comp(int l, int k, int d) {
  for (int i = 0, c = 0; i <= l; ++i)
    for (int j = 0; j <= i; ++j, ++c)
      if (c == k) return d == 0 ? l - i : d == 1 ? i - j : j;
  return 0;
}

// S and T blocks of one pair.
template <int LA, int LB>
__device__ __forceinline__ void oei_st_values(const QxOei& A, int sa, int sb) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2;
  double bs[NA * NB] = {}, bt[NA * NB] = {};
  OeiPos<double> a, b;
  oei_atom(A, A.sh.atom[sa], a);
  oei_atom(A, A.sh.atom[sb], b);
  for (int ia = A.sh.poff[sa]; ia < A.sh.poff[sa] + A.sh.nprim[sa]; ++ia)
    for (int ib = A.sh.poff[sb]; ib < A.sh.poff[sb] + A.sh.nprim[sb]; ++ib) {
      const OeiPrim<double> P = oei_prim<double>(A, a, b, ia, ib);
      double s[3][LA + 1][LB + 3];
      oei_s1d<LA, LB + 2>(P, s);
      const double q = QX_PI / P.p, pre = P.K * q * sqrt(q);
      double t[3][LA + 1][LB + 1];
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int i = 0; i <= LA; ++i)
#pragma unroll
          for (int j = 0; j <= LB; ++j) t[d][i][j] = oei_t1<LA, LB + 2>(s[d], P.b, i, j);
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int ax = oei_comp(LA, i, 0), ay = oei_comp(LA, i, 1), az = oei_comp(LA, i, 2);
          const int bx = oei_comp(LB, j, 0), by = oei_comp(LB, j, 1), bz = oei_comp(LB, j, 2);
          const double sx = s[0][ax][bx], sy = s[1][ay][by], sz = s[2][az][bz];
          bs[i * NB + j] += pre * sx * sy * sz;
          bt[i * NB + j] += pre * (t[0][ax][bx] * sy * sz + sx * t[1][ay][by] * sz + sx * sy * t[2][az][bz]);
        }
    }
  const int n = A.sh.ncart, ba = A.sh.bfc[sa], bb = A.sh.bfc[sb];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const size_t o = (size_t)(ba + i) * n + bb + j, r = (size_t)(bb + j) * n + ba + i;
      A.S[o] = bs[i * NB + j];
      A.T[o] = bt[i * NB + j];
      if (sa != sb) {
        A.S[r] = bs[i * NB + j];
        A.T[r] = bt[i * NB + j];
      }
    }
}

// Density block of a pair, both orders of a pair of different shells summed.
template <int NA, int NB>
__device__ __forceinline__ void oei_block(const double* D, int n, int ba, int bb, bool diag, double (&o)[NA * NB]) {
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      double v = D[(size_t)(ba + i) * n + bb + j];
      if (!diag) v += D[(size_t)(bb + j) * n + ba + i];
      o[i * NB + j] = v;
    }
}

// Overlap and kinetic derivative of one pair with respect to coordinate X of
// centre A (SIDE 0) or B (SIDE 1), contracted with Wd and Pd.
template <int LA, int LB, int SIDE, int X, typename R>
__device__ __forceinline__ double oei_st_grad(const QxOei& A, int sa, int sb) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2;
  constexpr int IM = LA + (SIDE == 0), JM = LB + (SIDE == 1);
  double pd[NA * NB], wd[NA * NB];
  oei_block<NA, NB>(A.Pd, A.sh.ncart, A.sh.bfc[sa], A.sh.bfc[sb], sa == sb, pd);
  oei_block<NA, NB>(A.Wd, A.sh.ncart, A.sh.bfc[sa], A.sh.bfc[sb], sa == sb, wd);
  OeiPos<R> a, b;
  oei_atom(A, A.sh.atom[sa], a);
  oei_atom(A, A.sh.atom[sb], b);
  double g = 0.0;
  for (int ia = A.sh.poff[sa]; ia < A.sh.poff[sa] + A.sh.nprim[sa]; ++ia)
    for (int ib = A.sh.poff[sb]; ib < A.sh.poff[sb] + A.sh.nprim[sb]; ++ib) {
      const OeiPrim<R> P = oei_prim<R>(A, a, b, ia, ib);
      R s[3][IM + 1][JM + 3];
      oei_s1d<IM, JM + 2>(P, s);
      const double q = QX_PI / P.p, ex2 = 2.0 * (SIDE == 0 ? P.a : P.b);
      const R pre = (q * sqrt(q)) * P.K;
      R t[3][LA + 1][LB + 1], ds[LA + 1][LB + 1], dt[LA + 1][LB + 1];
#pragma unroll
      for (int i = 0; i <= LA; ++i)
#pragma unroll
        for (int j = 0; j <= LB; ++j) {
#pragma unroll
          for (int d = 0; d < 3; ++d) t[d][i][j] = oei_t1<IM, JM + 2>(s[d], P.b, i, j);
          const int n = SIDE == 0 ? i : j, up0 = i + (SIDE == 0), up1 = j + (SIDE == 1);
          ds[i][j] = ex2 * s[X][up0][up1];
          dt[i][j] = ex2 * oei_t1<IM, JM + 2>(s[X], P.b, up0, up1);
          if (n > 0) {
            const int d0 = i - (SIDE == 0), d1 = j - (SIDE == 1);
            ds[i][j] = ds[i][j] - (double)n * s[X][d0][d1];
            dt[i][j] = dt[i][j] - (double)n * oei_t1<IM, JM + 2>(s[X], P.b, d0, d1);
          }
        }
      constexpr int Y = (X + 1) % 3, Z = (X + 2) % 3;
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int ax = oei_comp(LA, i, X), ay = oei_comp(LA, i, Y), az = oei_comp(LA, i, Z);
          const int bx = oei_comp(LB, j, X), by = oei_comp(LB, j, Y), bz = oei_comp(LB, j, Z);
          const R syz = s[Y][ay][by] * s[Z][az][bz];
          const R tyz = t[Y][ay][by] * s[Z][az][bz] + s[Y][ay][by] * t[Z][az][bz];
          const R dS = pre * (ds[ax][bx] * syz), dT = pre * (dt[ax][bx] * syz + ds[ax][bx] * tyz);
          g += pd[i * NB + j] * oei_out(dT) + wd[i * NB + j] * oei_out(dS);
        }
    }
  return g;
}

// Values of one class: grid row 0 attraction, row 1 overlap and kinetic.
// CORE adds one primitive and nucleus to the [e|0] sums, HRR transfers them.
template <int LA, int LB, int NS, class Core, class Hrr>
__device__ __forceinline__ void oei_values(const QxOei& A, Core core, Hrr hrr) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2;
  int sa, sb;
  if (blockIdx.y == 1) {
    const int t = blockIdx.x * QX_OEI_BLOCK + threadIdx.x;
    if (t >= A.npair) return;
    oei_pair(A, t, LA == LB, sa, sb);
    oei_st_values<LA, LB>(A, sa, sb);
    return;
  }
  const int t = (blockIdx.x * QX_OEI_BLOCK + threadIdx.x) / QX_OEI_LANES, lane = threadIdx.x % QX_OEI_LANES;
  const bool in = t < A.npair;
  double s[NS] = {};
  OeiPos<double> a{}, b{};
  sa = sb = 0;
  if (in) {
    oei_pair(A, t, LA == LB, sa, sb);
    oei_atom(A, A.sh.atom[sa], a);
    oei_atom(A, A.sh.atom[sb], b);
    for (int ia = A.sh.poff[sa]; ia < A.sh.poff[sa] + A.sh.nprim[sa]; ++ia)
      for (int ib = A.sh.poff[sb]; ib < A.sh.poff[sb] + A.sh.nprim[sb]; ++ib) {
        const OeiPrim<double> P = oei_prim<double>(A, a, b, ia, ib);
        const double pre = 2.0 * QX_PI / P.p * P.K;
        for (int at = lane; at < A.sh.natom; at += QX_OEI_LANES) {
          OeiPos<double> C;
          oei_atom(A, at, C);
          const double PC[3] = {P.P[0] - C.x[0], P.P[1] - C.x[1], P.P[2] - C.x[2]};
          double F[LA + LB + 1];
          qx_boys<LA + LB>(P.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), A.boys, F);
          const double f = -A.sh.Z[at] * pre;
#pragma unroll
          for (int m = 0; m <= LA + LB; ++m) F[m] *= f;
          core(P.PA, PC, P.oo2p, F, s);
        }
      }
  }
#pragma unroll
  for (int k = 0; k < NS; ++k)
#pragma unroll
    for (int off = QX_OEI_LANES / 2; off > 0; off >>= 1) s[k] += __shfl_xor(s[k], off);
  if (!in || lane != 0) return;
  double o[NA * NB];
  const double AB[3] = {a.x[0] - b.x[0], a.x[1] - b.x[1], a.x[2] - b.x[2]};
  hrr(AB, s, o);
  const int n = A.sh.ncart, ba = A.sh.bfc[sa], bb = A.sh.bfc[sb];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      A.V[(size_t)(ba + i) * n + bb + j] = o[i * NB + j];
      if (sa != sb) A.V[(size_t)(bb + j) * n + ba + i] = o[i * NB + j];
    }
}

// Gradient of one class: grid row 0 attraction (d/dC by translational
// invariance of each nucleus term), rows 1..6 overlap and kinetic.  Terms
// meet in LDS (contexts of up to QX_GRAD_LDS / 3 atoms) and reach the global
// gradient once per block.
template <int LA, int LB, typename R, class Core>
__device__ __forceinline__ void oei_grads(const QxOei& A, Core core) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2;
  __shared__ double sg[QX_GRAD_LDS];
  const int ng = 3 * A.sh.natom;
  const bool lds = ng <= QX_GRAD_LDS;
  if (lds) {
    for (int i = threadIdx.x; i < ng; i += QX_OEI_BLOCK) sg[i] = 0.0;
    __syncthreads();
  }
  auto add = [&](int slot, double v) {
    if (lds) atomicAdd(&sg[slot], v);
    else qx_atomic_add(&A.grad[slot], v);
  };
  int sa, sb;
  if (blockIdx.y > 0) {
    const int t = blockIdx.x * QX_OEI_BLOCK + threadIdx.x;
    if (t < A.npair) {
      oei_pair(A, t, LA == LB, sa, sb);
      double g = 0.0;
      switch (blockIdx.y) {  // block-uniform
        case 1: g = oei_st_grad<LA, LB, 0, 0, R>(A, sa, sb); break;
        case 2: g = oei_st_grad<LA, LB, 0, 1, R>(A, sa, sb); break;
        case 3: g = oei_st_grad<LA, LB, 0, 2, R>(A, sa, sb); break;
        case 4: g = oei_st_grad<LA, LB, 1, 0, R>(A, sa, sb); break;
        case 5: g = oei_st_grad<LA, LB, 1, 1, R>(A, sa, sb); break;
        default: g = oei_st_grad<LA, LB, 1, 2, R>(A, sa, sb); break;
      }
      const int k = blockIdx.y - 1;
      add(3 * A.sh.atom[k < 3 ? sa : sb] + k % 3, g);
    }
  } else {
    const int t = (blockIdx.x * QX_OEI_BLOCK + threadIdx.x) / QX_OEI_LANES, lane = threadIdx.x % QX_OEI_LANES;
    if (t < A.npair) {
      oei_pair(A, t, LA == LB, sa, sb);
      OeiPos<R> a, b;
      oei_atom(A, A.sh.atom[sa], a);
      oei_atom(A, A.sh.atom[sb], b);
      const R AB[3] = {a.x[0] - b.x[0], a.x[1] - b.x[1], a.x[2] - b.x[2]};
      double pd[NA * NB];
      oei_block<NA, NB>(A.Pd, A.sh.ncart, A.sh.bfc[sa], A.sh.bfc[sb], sa == sb, pd);
      double gt[6] = {};
      for (int at = lane; at < A.sh.natom; at += QX_OEI_LANES) {
        OeiPos<R> C;
        oei_atom(A, at, C);
        double g[6] = {};
        for (int ia = A.sh.poff[sa]; ia < A.sh.poff[sa] + A.sh.nprim[sa]; ++ia)
          for (int ib = A.sh.poff[sb]; ib < A.sh.poff[sb] + A.sh.nprim[sb]; ++ib) {
            const OeiPrim<R> P = oei_prim<R>(A, a, b, ia, ib);
            const R PC[3] = {P.P[0] - C.x[0], P.P[1] - C.x[1], P.P[2] - C.x[2]};
            R F[LA + LB + 2];
            oei_boys<LA + LB + 1>(P.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), A.boys, F);
            const R f = (-A.sh.Z[at] * 2.0 * QX_PI / P.p) * P.K;
#pragma unroll
            for (int m = 0; m <= LA + LB + 1; ++m) F[m] = f * F[m];
            core(P.PA, PC, P.oo2p, F, AB, 2.0 * P.a, 2.0 * P.b, pd, g);
          }
#pragma unroll
        for (int k = 0; k < 6; ++k) gt[k] += g[k];
#pragma unroll
        for (int x = 0; x < 3; ++x) add(3 * at + x, -(g[x] + g[3 + x]));
      }
      const int atA = A.sh.atom[sa], atB = A.sh.atom[sb];
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        add(3 * atA + x, gt[x]);
        add(3 * atB + x, gt[3 + x]);
      }
    }
  }
  if (lds) {
    __syncthreads();
    for (int i = threadIdx.x; i < ng; i += QX_OEI_BLOCK)
      if (sg[i] != 0.0) qx_atomic_add(&A.grad[i], sg[i]);
  }
}

// mode 0: S, T, V; 1: contracted gradient; 2: its derivative along tv
#define QX_DEFINE_OEI(NAME, LA, LB, NS)                                                           \
  __global__ __launch_bounds__(QX_OEI_BLOCK) void qx_k_oei_##NAME(QxOei A) {                      \
    oei_values<LA, LB, NS>(A, [](const double (&PA)[3], const double (&PC)[3], double o, const double (&F)[LA + LB + 1], \
                                 double (&s)[NS]) { qx_ov_##NAME<double>(PA, PC, o, F, s); },      \
                           [](const double (&AB)[3], const double (&s)[NS], double (&o)[NA_##NAME * NB_##NAME]) { \
                             qx_ovh_##NAME<double>(AB, s, o);                                     \
                           });                                                                    \
  }                                                                                               \
  template <typename R>                                                                           \
  __global__ __launch_bounds__(QX_OEI_BLOCK) void qx_k_oeig_##NAME(QxOei A) {                     \
    oei_grads<LA, LB, R>(A, [](const R (&PA)[3], const R (&PC)[3], double o, const R (&F)[LA + LB + 2], const R (&AB)[3], \
                               double wA, double wB, const double (&pd)[NA_##NAME * NB_##NAME], double (&g)[6]) { \
      qx_ovg_##NAME<R>(PA, PC, o, F, AB, wA, wB, pd, g);                                          \
    });                                                                                           \
  }                                                                                               \
  extern "C" int qx_launch_oei_##NAME(const QxOei* a, int mode, hipStream_t s) {                  \
    if (a->npair <= 0) return 0;                                                                  \
    const unsigned gx = (unsigned)(((long long)a->npair * QX_OEI_LANES + QX_OEI_BLOCK - 1) / QX_OEI_BLOCK); \
    if (mode == 0) hipLaunchKernelGGL(qx_k_oei_##NAME, dim3(gx, 2), dim3(QX_OEI_BLOCK), 0, s, *a); \
    else if (mode == 1) hipLaunchKernelGGL(qx_k_oeig_##NAME<double>, dim3(gx, 7), dim3(QX_OEI_BLOCK), 0, s, *a); \
    else hipLaunchKernelGGL(qx_k_oeig_##NAME<qx_dual>, dim3(gx, 7), dim3(QX_OEI_BLOCK), 0, s, *a); \
    return (int)hipGetLastError();                                                                \
  }
