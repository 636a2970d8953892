// Rys quadrature, several lanes per quartet: K and the adjoint gradient of the
// heavy classes, and every derivative tensor.
//
// A (dd|dd) quartet evaluated by one lane needs 961 [e0|f0] values and 216
// accumulators: 5-9 KB of scratch per lane, whose latency, not arithmetic,
// bounds the kernel.  Here NA * NB lanes of a wavefront share a quartet, one
// per bra function pair (as many quartets as fit share the wavefront):
//   1. one lane per (quartet, root, direction, power of b) runs the two-index
//      vertical recurrence and the horizontal transfers of that 1D integral
//      in registers and leaves its values in LDS;
//   2. each lane sums x * y * z over the roots for its (a, b) and all (c, d),
//      at most 36 values in registers, operands shared through LDS;
//   3. each lane contracts or stores its values.
// The two phases alternate within one wavefront, so no workgroup barrier
// separates them and the wavefronts of a CU hide each other's latency.  (With
// 128- or 256-lane groups and two barriers per step the (dd|dp) K kernel took
// 0.52-0.61 ms on the 280-function cluster, five times its arithmetic.)
// (Dupuis, Rys & King 1976; recurrences: Rys, Dupuis & King 1983.)
#pragma once
#include "qx_grad.h"
#include "qx_pairm.h"

// ---- roots and weights ------------------------------------------------------
// Per order N <= 6 the roots u = t^2 and weights of exp(-T t^2) on [0, 1], as
// degree-12 polynomials on unit intervals of T below QX_RYS_TMAX; above, the
// scaled half-range Hermite rule (the tail beyond t = 1 is below 1e-20).
#define QX_RYS_TMAX 72
#define QX_RYS_DEG 12
#define QX_RYS_NC (QX_RYS_DEG + 1)
#define QX_RYS_MAXN 6
// doubles of the tables of all orders below N, each 2 N (72 * 13 + 1)
__host__ __device__ constexpr int qx_rys_off(int N) { return N * (N - 1) * (QX_RYS_TMAX * QX_RYS_NC + 1); }
#define QX_RYS_DOUBLES (QX_RYS_MAXN * (QX_RYS_MAXN + 1) * (QX_RYS_TMAX * QX_RYS_NC + 1))

// Root r and its weight, with their derivative along the tangent for duals
// (the rule is exact for every T, so differentiating it is exact too).
template <int N>
__device__ __forceinline__ void qx_rys(const double* __restrict__ tab, double T, int r, double& u, double& w) {
  tab += qx_rys_off(N);
  if (T < (double)QX_RYS_TMAX) {
    const int iv = (int)T;
    const double x = 2.0 * (T - iv) - 1.0;
    const double* a = tab + (iv * 2 * N + r) * QX_RYS_NC;
    const double* b = a + N * QX_RYS_NC;
    double s = a[QX_RYS_DEG], t = b[QX_RYS_DEG];
#pragma unroll
    for (int k = QX_RYS_DEG - 1; k >= 0; --k) {
      s = s * x + a[k];
      t = t * x + b[k];
    }
    u = s;
    w = t;
  } else {
    const double* a = tab + QX_RYS_TMAX * 2 * N * QX_RYS_NC;
    const double o = 1.0 / T;
    u = a[r] * o;
    w = a[N + r] * sqrt(o);
  }
}
template <int N>
__device__ __forceinline__ void qx_rys(const double* __restrict__ tab, qx_dual T, int r, qx_dual& u, qx_dual& w) {
  tab += qx_rys_off(N);
  if (T.v < (double)QX_RYS_TMAX) {
    const int iv = (int)T.v;
    const double x = 2.0 * (T.v - iv) - 1.0;
    const double* a = tab + (iv * 2 * N + r) * QX_RYS_NC;
    const double* b = a + N * QX_RYS_NC;
    double s = a[QX_RYS_DEG], t = b[QX_RYS_DEG], ds = 0.0, dt = 0.0;
#pragma unroll
    for (int k = QX_RYS_DEG - 1; k >= 0; --k) {
      ds = ds * x + s;
      dt = dt * x + t;
      s = s * x + a[k];
      t = t * x + b[k];
    }
    u = qx_dual(s, 2.0 * ds * T.d);
    w = qx_dual(t, 2.0 * dt * T.d);
  } else {
    const double* a = tab + QX_RYS_TMAX * 2 * N * QX_RYS_NC;
    const double o = 1.0 / T.v, lu = a[r] * o, lw = a[N + r] * sqrt(o);
    u = qx_dual(lu, -lu * o * T.d);
    w = qx_dual(lw, -0.5 * lw * o * T.d);
  }
}

#define QX_INLINE __attribute__((always_inline))

// ---- 1D integrals -----------------------------------------------------------
template <typename R>
struct QxCoef {  // the type of a small integer factor
  using T = double;
};
template <>
struct QxCoef<float> {
  using T = float;
};

// Ix(i, j, k, l), i <= IA, k <= KC, l <= LD, of one root and direction into
// o[(i * (JB+1) + j) * NKS + k * (LD+1) + l], for one j <= JB or (ALL) every j.
template <int IA, int JB, int KC, int LD, int NKS, bool ALL, typename R>
__device__ __forceinline__ void qx_rys_1d(R start, R c0, R d0, R b10, R b01, R b00, R ab, R cd, int j, R* o) {
  using F = typename QxCoef<R>::T;
  constexpr int NM = IA + JB, MM = KC + LD;
  R g[NM + 1][MM + 1];
#pragma unroll
  for (int n = 0; n <= NM; ++n) {
    if (n == 0) g[0][0] = start;
    else if (n == 1) g[n][0] = c0 * g[0][0];
    else g[n][0] = c0 * g[n - 1][0] + F(n - 1) * b10 * g[n > 1 ? n - 2 : 0][0];
#pragma unroll
    for (int m = 1; m <= MM; ++m) {
      R v = d0 * g[n][m - 1];
      if (m > 1) v = v + F(m - 1) * b01 * g[n][m > 1 ? m - 2 : 0];
      if (n > 0) v = v + F(n) * b00 * g[n > 0 ? n - 1 : 0][m - 1];
      g[n][m] = v;
    }
  }
  // (i, j) = sum_k binomial(j, k) ab^(j-k) (i + k)
#pragma unroll
  for (int jj = 0; jj <= (ALL ? JB : 0); ++jj) {
    if (ALL) j = jj;
    const R t0 = j == 0 ? R(1) : j == 1 ? ab : ab * ab;
    const R t1 = j == 0 ? R(0) : j == 1 ? R(1) : F(2) * ab;
    const R t2 = j == 2 ? R(1) : R(0);
    R* const oj = o + j * NKS;
#pragma unroll
    for (int i = 0; i <= IA; ++i) {
      R k[MM + 1];
#pragma unroll
      for (int m = 0; m <= MM; ++m) {
        if (JB == 0 || (ALL && jj == 0)) k[m] = g[i][m];
        else if (ALL && jj == 1) k[m] = ab * g[i][m] + g[i + 1 <= NM ? i + 1 : 0][m];
        else if (JB == 1) k[m] = t0 * g[i][m] + t1 * g[i + 1 <= NM ? i + 1 : 0][m];
        else k[m] = t0 * g[i][m] + t1 * g[i + 1 <= NM ? i + 1 : 0][m] + t2 * g[i + 2 <= NM ? i + 2 : 0][m];
      }
#pragma unroll
      for (int l = 0; l <= LD; ++l) {
        if (l > 0) {
#pragma unroll
          for (int m = 0; m <= MM - l; ++m) k[m] = k[m + 1] + cd * k[m];
        }
#pragma unroll
        for (int kk = 0; kk <= KC; ++kk) oj[i * (JB + 1) * NKS + kk * (LD + 1) + l] = k[kk];
      }
    }
  }
}

// One primitive pair's geometry and its shell pair's first centre and A - B.
template <typename G>
struct QxRysPair {
  double p;
  G K, P[3], A[3], AB[3];
};
__device__ __forceinline__ void qx_rys_pair(const QxArgs& A_, int P, int u, QxRysPair<double>& r) {
  r.p = A_.pp.p[u];
  r.K = A_.pp.K[u];
  r.P[0] = A_.pp.Px[u]; r.P[1] = A_.pp.Py[u]; r.P[2] = A_.pp.Pz[u];
  r.A[0] = A_.pr.Ax[P]; r.A[1] = A_.pr.Ay[P]; r.A[2] = A_.pr.Az[P];
  r.AB[0] = A_.pr.ABx[P]; r.AB[1] = A_.pr.ABy[P]; r.AB[2] = A_.pr.ABz[P];
}
__device__ __forceinline__ void qx_rys_pair(const QxArgs& A_, int P, int u, QxRysPair<qx_dual>& r) {
  const QxTanPair t = qx_tan_pair(A_, P, u);
  r.p = A_.pp.p[u];
  r.K = t.K;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r.P[d] = t.P[d];
    r.A[d] = t.A[d];
    r.AB[d] = t.AB[d];
  }
}
__device__ __forceinline__ void qx_rys_cast(double x, double& o) { o = x; }
__device__ __forceinline__ void qx_rys_cast(double x, float& o) { o = (float)x; }
__device__ __forceinline__ void qx_rys_cast(qx_dual x, qx_dual& o) { o = x; }

// Recurrence parameters of one (quartet, root): c0 and d0 per direction, b10,
// b01, b00, the weight with all prefactors, and C - D.
#define QX_RYS_PAR 13
template <int N, typename G, typename R>
__device__ __forceinline__ void qx_rys_params(const QxArgs& A_, const double* tab, int P1, int u1, int P2, int u2, int root,
                                              R (&o)[QX_RYS_PAR]) {
  QxRysPair<G> b, k;
  qx_rys_pair(A_, P1, u1, b);
  qx_rys_pair(A_, P2, u2, k);
  const double p = b.p, q = k.p;
  const double pq = p + q, rs = 1.0 / sqrt(pq), opq = rs * rs, oo = 0.5 / (p * q);  // 1/2p = q oo, 1/2q = p oo
  G X[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) X[d] = b.P[d] - k.P[d];
  G u, w;
  qx_rys<N>(tab, (p * q * opq) * (X[0] * X[0] + X[1] * X[1] + X[2] * X[2]), root, u, w);
  const G fu = opq * u, qf = q * fu, pf = p * fu;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    qx_rys_cast(b.P[d] - b.A[d] - qf * X[d], o[d]);
    qx_rys_cast(k.P[d] - k.A[d] + pf * X[d], o[3 + d]);
    qx_rys_cast(k.AB[d], o[10 + d]);
  }
  qx_rys_cast((q * oo) * (1.0 - qf), o[6]);
  qx_rys_cast((p * oo) * (1.0 - pf), o[7]);
  qx_rys_cast(0.5 * fu, o[8]);
  qx_rys_cast((2.0 * QX_TWO_PI_5_2 * oo * rs) * (w * (b.K * k.K)), o[9]);
}

// Shapes of the kernels of one class; DER = 1 raises a and c by one.
// Wavefronts work alone, so a block is any number of them: 4, or 8 where the
// K' rows leave a CU room for one block only.
#define QX_RYS_BLOCK 256
// LDS values per wavefront: 19 KB in FP64, so that two blocks of four share a CU
#define QX_RYS_LDS 2464
#define QX_RYS_BLOCK_MAX 512
template <int LA, int LB, int LC, int LD, int DER>
struct QxRys {
  static constexpr int NA = qx_ncart(LA), NB = qx_ncart(LB), NC = qx_ncart(LC), ND = qx_ncart(LD);
  static constexpr int N = (LA + LB + LC + LD + DER) / 2 + 1;
  static constexpr int G = NA * NB;                       // lanes per quartet
  static constexpr int IA = LA + DER, KC = LC + DER;
  static constexpr int NKL = (KC + 1) * (LD + 1);
  static constexpr int NKS = NKL | 1;                     // stride of the (i, j) rows, odd against bank conflicts
  static constexpr int NKU = (LC + 1) * (LD + 1);         // of an undifferentiated ket
  static constexpr int NG = (IA + 1) * (LB + 1) * NKS;    // 1D values per root and direction
  static constexpr int STRIDE = (3 * N * NG) | 1;         // per quartet, odd against bank conflicts
  static constexpr int ONE = STRIDE + QX_RYS_PAR * N;     // LDS values of one quartet
  // quartets per wavefront: as many as its lanes hold and QX_RYS_LDS values allow
  static constexpr int FIT = QX_RYS_LDS / ONE < 1 ? 1 : QX_RYS_LDS / ONE;
  static constexpr int Q = 64 / G < FIT ? 64 / G : FIT;
  static constexpr int SUM = (Q * G) | 1;                 // row stride of the sums over a quartet's lanes
  static constexpr int SUMS = 2 * (DER ? 6 : NC + ND) * SUM;  // their LDS values (FP32: two per sum)
  static constexpr int LDS = Q * ONE > SUMS ? (Q * ONE + 1) & ~1 : SUMS;  // values per wavefront
  // 1D tasks: one per power of b, or all of them where that fits one pass of the wavefront better
  static constexpr bool ALLJ = LB > 0 && 3 * Q * N * (LB + 1) > 64 && 3 * Q * N <= 64;
  static constexpr int TASKS = 3 * N * (ALLJ ? 1 : LB + 1);  // per quartet
  static constexpr int SETS = Q * N;                      // parameter sets of one step
  static constexpr int STEPS = 64 / SETS;                 // steps whose sets one wavefront holds
  static_assert(STEPS >= 1, "parameter sets of a step");
  // four wavefronts in dual numbers (16 bytes) and the gradient's accumulators fit a workgroup's 160 KB
  static_assert(4 * 16 * LDS + 8 * QX_GRAD_LDS <= 160 * 1024, "LDS of a quadrature workgroup");
};

// Orders a wavefront's own LDS writes before its reads (and back): its lanes
// run in step and LDS serves one wavefront in order, so only the compiler has
// to be held.
__device__ __forceinline__ void qx_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Most primitives of the kets in flight (wave-uniform).
__device__ __forceinline__ int qx_rys_prims(const QxArgs& A_, int pk0, int nq) {
  int n = 1;
  for (int q = 0; q < nq; ++q) n = max(n, A_.pr.pp_n[pk0 + q]);
  return n;
}

// Runs the wavefront's share of a block's kets, Q at a time: begin(first ket,
// how many), per primitive quartet step(i1, i2) with the 1D integrals at g,
// end().  Every lane of the wavefront calls all three.  Workgroups of one grid
// column share the primitive quartets: the few long sums of a small contracted
// molecule would otherwise run one after the other in a handful of wavefronts.
//
// Roots, weights and recurrence parameters of STEPS steps ahead (of several
// ket groups, or for contracted pairs of several primitive quartets) are
// worked out at once, one lane per (step, quartet, root), and kept in that
// lane's registers: their chain of loads (pair, primitive, table row) and the
// root polynomials would otherwise be waited for in every step, with a
// handful of lanes busy.  A step's lanes then hand them to the 1D tasks
// through LDS.  (Read by every 1D task itself, those loads kept the CU's
// address unit busy four times longer than the arithmetic took; one step at a
// time, (dd|ps) of a 280-function gradient took 1.22 ms against 1.08 so.)
template <class S, int LB, int LD, typename G, typename R, bool SHARE, class Begin, class Step, class End>
__device__ __forceinline__ void qx_rys_walk(const QxArgs& A_, const QxKList& kl, const QxKBlock& b, R* g, Begin begin, Step step,
                                            End end) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int u1 = A_.pr.pp_first[b.P1], n1 = A_.pr.pp_n[b.P1];
  QxRysPair<G> bra;
  qx_rys_pair(A_, b.P1, u1, bra);
  R ab[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) qx_rys_cast(bra.AB[d], ab[d]);
  R* const par = g + S::Q * S::STRIDE;
  const bool single = n1 == 1 && kl.ketprim == 1;
  const int share = ((b.j1 - b.j0 + S::Q - 1) / S::Q + waves - 1) / waves * S::Q;
  const int k0 = b.j0 + wave * share, k1 = min(b.j1, k0 + share);
  const int ps = lane / S::SETS, pe = lane - ps * S::SETS, pq = pe / S::N, pr = pe - pq * S::N;  // the lane's set
  R pv[QX_RYS_PAR];
#pragma unroll
  for (int i = 0; i < QX_RYS_PAR; ++i) pv[i] = R(0.0);
  int held = 0;  // the step whose sets are next, single primitives
  for (int k = k0; k < k1; k += S::Q) {
    const int nq = min(S::Q, k1 - k), pk0 = b.kst + k;
    // the workgroup's share of the primitive quartets
    const int n2 = kl.ketprim > 1 ? qx_rys_prims(A_, pk0, nq) : 1;
    int mb = 0, nc = n1 * n2;
    if (SHARE && kl.psplit > 1) {
      const long long all = nc;
      mb = (int)(all * blockIdx.z / kl.psplit);
      nc = (int)(all * (blockIdx.z + 1) / kl.psplit);
      if (mb >= nc) continue;
    }
    begin(pk0, nq);
    for (int m = mb; m < nc; ++m) {
      const int now = single ? held : (m - mb) % S::STEPS;
      if (now == 0) {
        const int m1 = m + ps, i1 = single ? 0 : m1 / n2, i2 = single ? 0 : m1 - i1 * n2;
        const int P2 = pk0 + (single ? ps * S::Q : 0) + pq;
        if (ps < S::STEPS && (single ? P2 < b.kst + k1 : pq < nq && m1 < nc) && i2 < A_.pr.pp_n[min(P2, b.kst + k1 - 1)])
          qx_rys_params<S::N, G, R>(A_, kl.rys, b.P1, u1 + i1, P2, A_.pr.pp_first[P2] + i2, pr, pv);
      }
      held = now + 1 < S::STEPS ? now + 1 : 0;
      qx_wave_sync();  // the previous step's values have been read
      if (ps == now) {
#pragma unroll
        for (int i = 0; i < QX_RYS_PAR; ++i) par[pe * QX_RYS_PAR + i] = pv[i];
      }
      qx_wave_sync();
      for (int t = lane; t < nq * S::TASKS; t += 64) {
        constexpr int J = S::ALLJ ? 1 : LB + 1;
        const int q = t / S::TASKS, rdj = t - q * S::TASKS, rd = rdj / J, r = rd / 3, dim = rd - 3 * r;
        const R* o = par + (q * S::N + r) * QX_RYS_PAR;
        qx_rys_1d<S::IA, LB, S::KC, LD, S::NKS, S::ALLJ, R>(
            dim == 0 ? o[9] : R(1), o[dim], o[3 + dim], o[6], o[7], o[8], dim == 0 ? ab[0] : dim == 1 ? ab[1] : ab[2],
            o[10 + dim], rdj - rd * J, g + q * S::STRIDE + rd * S::NG);
      }
      qx_wave_sync();
      step(m / n2, m - m / n2 * n2);
    }
    end();
  }
}

// The lane's bra function pair and quartet slot; exponents of (a, b) per direction.
template <class S, int LA, int LB>
struct QxRysLane {
  int slot, ab, ca, cb, e[3][2];
  bool in;
  __device__ __forceinline__ QxRysLane() {
    slot = (threadIdx.x & 63) / S::G;
    ab = (threadIdx.x & 63) % S::G;
    ca = ab / S::NB;
    cb = ab % S::NB;
    in = slot < S::Q;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      e[d][0] = e[d][1] = 0;
#pragma unroll
      for (int i = 0; i < S::NA; ++i) e[d][0] = i == ca ? qx_comp(LA, i, d) : e[d][0];
#pragma unroll
      for (int j = 0; j < S::NB; ++j) e[d][1] = j == cb ? qx_comp(LB, j, d) : e[d][1];
    }
  }
  __device__ __forceinline__ int off(int d) const { return (e[d][0] * (LB + 1) + e[d][1]) * S::NKS; }
};

// I[c][d] += the lane's integrals of one primitive quartet.
template <class S, int LC, int LD, typename R, typename T>
__device__ __forceinline__ void qx_rys_sum(const R* gq, int ox, int oy, int oz, T (&I)[S::NC * S::ND]) {
#pragma unroll 1
  for (int r = 0; r < S::N; ++r) {
    R x[S::NKL], y[S::NKL], z[S::NKL];
#pragma unroll
    for (int k = 0; k < S::NKL; ++k) {
      x[k] = gq[(3 * r + 0) * S::NG + ox + k];
      y[k] = gq[(3 * r + 1) * S::NG + oy + k];
      z[k] = gq[(3 * r + 2) * S::NG + oz + k];
    }
#pragma unroll
    for (int c = 0; c < S::NC; ++c)
#pragma unroll
      for (int d = 0; d < S::ND; ++d)
        I[c * S::ND + d] += T(x[qx_comp(LC, c, 0) * (LD + 1) + qx_comp(LD, d, 0)] *
                              y[qx_comp(LC, c, 1) * (LD + 1) + qx_comp(LD, d, 1)] *
                              z[qx_comp(LC, c, 2) * (LD + 1) + qx_comp(LD, d, 2)]);
  }
}

// ---- K ------------------------------------------------------------------------
// Bound by LDS (busy 51-54 % of the cycles) and latency at two or three
// wavefronts per SIMD (FP64 issue 17-26 %).  K'_a then K'_b: a lane's sums over (c, d) are added
// over its quartet's lanes in LDS, one atomic per row element instead of one
// per lane ((dd|dp) of 280 functions 457 -> 357 us, (dp|dp) 403 -> 336, with
// larger shares of kets per workgroup 322 and 291).
// SHARE: workgroups share primitive quartets (a kernel of its own: as a branch,
// the walk's longer index arithmetic cost 1.3 % where there is one).
template <int LA, int LB, int LC, int LD, typename G, typename R, bool ROWS, bool STAGE, bool SHARE>
__global__ __launch_bounds__(QX_RYS_BLOCK_MAX) void qx_rk(QxArgs A_, QxKList kl) {
  using S = QxRys<LA, LB, LC, LD, 0>;
  constexpr int NA = S::NA, NB = S::NB, NC = S::NC, ND = S::ND;
  HIP_DYNAMIC_SHARED(double, qx_sk)
  QxKBlock b;
  if (!qx_k_block(A_, kl, b)) return;
  R* const g = reinterpret_cast<R*>(qx_sk + (ROWS ? (STAGE ? 2 : 1) * (NA + NB) * b.W : 0)) + (threadIdx.x >> 6) * S::LDS;
  if (ROWS) qx_k_rows_begin<NA, NB, STAGE>(A_, b, qx_sk);
  const QxRysLane<S, LA, LB> ln;
  const int n = A_.e.nbf, ca = ln.ca, cb = ln.cb;
  const int ia = A_.pr.bfa[b.P1], ib = A_.pr.bfb[b.P1];
  bool act = false;
  int P2 = 0, pk = 0, nk = 0;
  G I[NC * ND];
  qx_rys_walk<S, LB, LD, G, R, SHARE>(
      A_, kl, b, g,
      [&](int pk0, int nq) QX_INLINE {
        pk = pk0;
        nk = nq;
        act = ln.in && ln.slot < nq;
        P2 = pk0 + (act ? ln.slot : 0);
#pragma unroll
        for (int k = 0; k < NC * ND; ++k) I[k] = G(0.0);
      },
      [&](int, int i2) QX_INLINE {
        if (act && i2 < A_.pr.pp_n[P2])
          qx_rys_sum<S, LC, LD>(g + ln.slot * S::STRIDE, ln.off(0), ln.off(1), ln.off(2), I);
      },
      [&]() QX_INLINE {
        static_assert((NC + ND) * S::SUM * sizeof(double) <= S::LDS * sizeof(R), "LDS of the lane sums");
        double* const sum = reinterpret_cast<double*>(g);
        const double fk = act ? 2.0 * qx_degeneracy(A_, b.P1, P2) : 0.0;
        const int ic = A_.pr.bfa[P2], id = A_.pr.bfb[P2], lane = threadIdx.x & 63;
#pragma unroll
        for (int side = 0; side < 2; ++side) {  // K'_a from D_b, then K'_b from D_a
          double v[NC + ND] = {};
          if (act) {
            const double* dx;
            if (STAGE) dx = qx_sk + (side == 0 ? NA + NB + NA + cb : NA + NB + ca) * b.W - b.col0;
            else dx = A_.e.D + (size_t)(side == 0 ? ib + cb : ia + ca) * n;
            double xd[ND];
#pragma unroll
            for (int d = 0; d < ND; ++d) xd[d] = fk * dx[id + d];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              const double xc = fk * dx[ic + c];
#pragma unroll
              for (int d = 0; d < ND; ++d) {
                const double t = qx_value(I[c * ND + d]);
                v[c] += t * xd[d];
                v[NC + d] += t * xc;
              }
            }
          }
          qx_wave_sync();
          if (act) {
#pragma unroll
            for (int x = 0; x < NC + ND; ++x) sum[x * S::SUM + ln.slot * S::G + ln.ab] = v[x];
          }
          qx_wave_sync();
          const int own = side == 0 ? NA : NB, len = side == 0 ? NB : NA;
          for (int t = lane; t < nk * own * (NC + ND); t += 64) {
            const int q = t / (own * (NC + ND)), cx = t - q * own * (NC + ND), o = cx / (NC + ND), x = cx - o * (NC + ND);
            const double* w = sum + x * S::SUM + q * S::G + o * (side == 0 ? NB : 1);
            double r = 0.0;
#pragma unroll
            for (int k = 0; k < len; ++k) r += w[k * (side == 0 ? 1 : NB)];
            const int col = x < NC ? A_.pr.bfa[pk + q] + x : A_.pr.bfb[pk + q] + x - NC;
            if (ROWS) atomicAdd(qx_sk + (side == 0 ? o : NA + o) * b.W + col - b.col0, r);
            else qx_atomic_add(A_.e.K + (size_t)((side == 0 ? ia : ib) + o) * n + col, r);
          }
        }
      });
  if (ROWS) qx_k_rows_end<NA, NB>(A_, b, qx_sk);
}

// ---- integrals and derivative integrals into the pair matrix --------------------
// TO: 0 into the matrix; 1 added to it, where workgroups share primitive
// quartets; 2 into the class-blocked array of a single-primitive basis.  (A
// choice per launch: as branches of one kernel it cost (dp|dp) 20 %.)
template <int LA, int LB, int LC, int LD, int TO>
__global__ __launch_bounds__(QX_RYS_BLOCK) void qx_re(QxArgs A_, QxKList kl, QxPairM pm) {
  using S = QxRys<LA, LB, LC, LD, 0>;
  HIP_DYNAMIC_SHARED(double, qx_sk)
  QxKBlock b;
  if (!qx_k_block(A_, kl, b)) return;
  double* const g = qx_sk + (threadIdx.x >> 6) * S::LDS;
  const QxRysLane<S, LA, LB> ln;
  bool act = false;
  int P2 = 0;
  double I[S::NC * S::ND];
  qx_rys_walk<S, LB, LD, double, double, TO == 1>(
      A_, kl, b, g,
      [&](int pk0, int nq) QX_INLINE {
        act = ln.in && ln.slot < nq;
        P2 = pk0 + (act ? ln.slot : 0);
#pragma unroll
        for (int k = 0; k < S::NC * S::ND; ++k) I[k] = 0.0;
      },
      [&](int, int i2) QX_INLINE {
        if (act && i2 < A_.pr.pp_n[P2])
          qx_rys_sum<S, LC, LD>(g + ln.slot * S::STRIDE, ln.off(0), ln.off(1), ln.off(2), I);
      },
      [&]() QX_INLINE {
        if (act && !(A_.e.skip_single && qx_single_atom(A_, b.P1, P2))) {
          if (TO == 2) {
            double* m = A_.e.out + A_.w.store_base + (long long)ln.ab * (S::NC * S::ND) * kl.nquart + kl.prefix[blockIdx.x] +
                        (P2 - b.kst);
#pragma unroll
            for (int k = 0; k < S::NC * S::ND; ++k) m[k * kl.nquart] = I[k];
            return;
          }
          double* m = pm.M + (pm.row0 + b.P1 - pm.rowp + (long long)ln.ab * pm.rown) * pm.ld + pm.col0 + (P2 - pm.colp);
#pragma unroll
          for (int k = 0; k < S::NC * S::ND; ++k) {
            if (TO == 1) qx_atomic_add(&m[(long long)k * pm.coln], I[k]);
            else m[(long long)k * pm.coln] = I[k];
          }
        }
      });
}

// The Schwarz pass: (ab|ab) of every pair, one wavefront each, by pair and
// function pair.
template <int LA, int LB>
__global__ __launch_bounds__(64) void qx_rs(QxArgs A_, QxKList kl) {
  using S = QxRys<LA, LB, LA, LB, 0>;
  HIP_DYNAMIC_SHARED(double, qx_sk)
  const int P = kl.bra0 + (int)blockIdx.x;
  const QxKBlock b{P, 0, 1, P, 0, 0};
  const QxRysLane<S, LA, LB> ln;
  double I[S::NC * S::ND] = {};
  qx_rys_walk<S, LB, LB, double, double, false>(
      A_, kl, b, qx_sk, [&](int, int) QX_INLINE {},
      [&](int, int) QX_INLINE {
        if (ln.slot == 0) qx_rys_sum<S, LA, LB>(qx_sk, ln.off(0), ln.off(1), ln.off(2), I);
      },
      [&]() QX_INLINE {
        if (ln.slot != 0) return;
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < S::NC * S::ND; ++k) v = k == ln.ab ? I[k] : v;
        A_.e.out[(long long)P * QX_PAIR_STRIDE + ln.ab] = v;
      });
}

// Values of one direction for the lane's (a, b), ket index k and all l: the
// integral (o), d/dA (a), d/dB (b) and d/dC (c) factors.
template <class S, int LB, int LD, typename R>
struct QxRysRow {
  R o[LD + 1], a[LD + 1], b[LD + 1], c[LD + 1];
};
template <class S, int LB, int LD, typename R, typename F>
__device__ __forceinline__ void qx_rys_row(const R* gd, int i, int j, int k, R ab, F wa, F wb, F wc,
                                           QxRysRow<S, LB, LD, R>& r) {
  const R* o = gd + (i * (LB + 1) + j) * S::NKS + k * (LD + 1);
  const R* up = o + (LB + 1) * S::NKS;
  const R* dn = o - (i > 0 ? (LB + 1) * S::NKS : 0);
  const R* bj = o - (j > 0 ? S::NKS : 0);
  const R* kd = o - (k > 0 ? LD + 1 : 0);
#pragma unroll
  for (int l = 0; l <= LD; ++l) {
    const R u = up[l];
    r.o[l] = o[l];
    r.a[l] = wa * u - F(i) * dn[l];
    r.b[l] = wb * (u + ab * r.o[l]) - F(j) * bj[l];
    r.c[l] = wc * o[LD + 1 + l] - F(k) * kd[l];
  }
}

// First-derivative integrals into the slices of the coordinates (G = qx_dual:
// their derivatives along tv).  One ket c component at a time keeps the nine
// derivative values of its d components in registers; contracted quartets add
// up in the matrix, by atomics that no step waits for.
template <int LA, int LB, int LC, int LD, typename G>
__global__ __launch_bounds__(QX_RYS_BLOCK) void qx_rd(QxArgs A_, QxKList kl, QxPairM pm) {
  using S = QxRys<LA, LB, LC, LD, 1>;
  constexpr int ND = S::ND;
  HIP_DYNAMIC_SHARED(double, qx_sk)
  G* const g = reinterpret_cast<G*>(qx_sk) + (threadIdx.x >> 6) * S::LDS;
  QxKBlock b;
  if (!qx_k_block(A_, kl, b)) return;
  const QxRysLane<S, LA, LB> ln;
  const int u1 = A_.pr.pp_first[b.P1], prims = A_.pr.pp_n[b.P1] * kl.ketprim;
  G ab[3];
  {
    QxRysPair<G> bra;
    qx_rys_pair(A_, b.P1, u1, bra);
#pragma unroll
    for (int d = 0; d < 3; ++d) ab[d] = bra.AB[d];
  }
  bool act = false;
  int P2 = 0, at[4];
  qx_rys_walk<S, LB, LD, G, G, true>(
      A_, kl, b, g,
      [&](int pk0, int nq) QX_INLINE {
        const bool in = ln.in && ln.slot < nq;
        P2 = pk0 + (in ? ln.slot : 0);
        act = in && !qx_single_atom(A_, b.P1, P2);
        at[0] = A_.pr.atom_a[b.P1]; at[1] = A_.pr.atom_b[b.P1]; at[2] = A_.pr.atom_a[P2]; at[3] = A_.pr.atom_b[P2];
      },
      [&](int i1, int i2) QX_INLINE {
        if (!act || i2 >= A_.pr.pp_n[P2]) return;
        double* const m = pm.M + (pm.row0 + b.P1 - pm.rowp + (long long)ln.ab * pm.rown) * pm.ld + pm.col0 + (P2 - pm.colp);
        const double wa = A_.pp.a2[u1 + i1], wb = A_.pp.b2[u1 + i1], wc = A_.pp.a2[A_.pr.pp_first[P2] + i2];
        const G* gq = g + ln.slot * S::STRIDE;
#pragma unroll 1
        for (int c = 0; c < S::NC; ++c) {
          int kx = 0, ky = 0, kz = 0;
#pragma unroll
          for (int k = 0; k < S::NC; ++k) {
            kx = k == c ? qx_comp(LC, k, 0) : kx;
            ky = k == c ? qx_comp(LC, k, 1) : ky;
            kz = k == c ? qx_comp(LC, k, 2) : kz;
          }
          G v[9][ND];
#pragma unroll
          for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int d = 0; d < ND; ++d) v[t][d] = G(0.0);
#pragma unroll 1
          for (int r = 0; r < S::N; ++r) {
            QxRysRow<S, LB, LD, G> x, y, z;
            qx_rys_row<S, LB, LD, G, double>(gq + (3 * r + 0) * S::NG, ln.e[0][0], ln.e[0][1], kx, ab[0], wa, wb, wc, x);
            qx_rys_row<S, LB, LD, G, double>(gq + (3 * r + 1) * S::NG, ln.e[1][0], ln.e[1][1], ky, ab[1], wa, wb, wc, y);
            qx_rys_row<S, LB, LD, G, double>(gq + (3 * r + 2) * S::NG, ln.e[2][0], ln.e[2][1], kz, ab[2], wa, wb, wc, z);
#pragma unroll
            for (int d = 0; d < ND; ++d) {
              const int lx = qx_comp(LD, d, 0), ly = qx_comp(LD, d, 1), lz = qx_comp(LD, d, 2);
              const G yz = y.o[ly] * z.o[lz], xz = x.o[lx] * z.o[lz], xy = x.o[lx] * y.o[ly];
              v[0][d] += x.a[lx] * yz; v[1][d] += y.a[ly] * xz; v[2][d] += z.a[lz] * xy;
              v[3][d] += x.b[lx] * yz; v[4][d] += y.b[ly] * xz; v[5][d] += z.b[lz] * xy;
              v[6][d] += x.c[lx] * yz; v[7][d] += y.c[ly] * xz; v[8][d] += z.c[lz] * xy;
            }
          }
#pragma unroll
          for (int ce = 0; ce < 4; ++ce) {
            bool lead = true;  // the first centre of its atom stores the atom's sum
            double f[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              if (k < ce) lead = lead && at[k] != at[ce];
              else f[k] = at[k] == at[ce] ? 1.0 : 0.0;
            }
            if (!lead) continue;
            const double f0 = f[0] - f[3], f1 = f[1] - f[3], f2 = f[2] - f[3];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              const long long sl = qx_dfull_slice(A_.e, 3 * at[ce] + x);
              if (sl < 0) continue;
              double* o = m + sl * pm.slice + (long long)c * ND * pm.coln;
#pragma unroll
              for (int d = 0; d < ND; ++d) {
                const double s = f0 * qx_value(v[x][d]) + f1 * qx_value(v[3 + x][d]) + f2 * qx_value(v[6 + x][d]);
                if (prims > 1) qx_atomic_add(&o[(long long)d * pm.coln], s);
                else o[(long long)d * pm.coln] = s;
              }
            }
          }
        }
      },
      [&]() QX_INLINE {});
}

// ---- adjoint gradient ------------------------------------------------------------
// 8 f Gamma_abcd, Gamma = 2 D_ab D_cd - (D_ac D_bd + D_ad D_bc) / 2, for the
// lane's (a, b) and every (c, d); summed against the derivative integrals.
// Per root the sum over (c, d) goes to the adjoint of each direction's 1D
// values first (w: 5 multiply-adds per (c, d)), which then meets the raised
// and lowered values: the nine derivative values per (c, d) are never formed
// ((dd|dp) of 280 functions: 1.77 ms at one wavefront per SIMD -> 0.98 at two).
// Bound by LDS reads (busy 52-68 % of the cycles) and VALU issue (41-53 %) at two wavefronts per
// SIMD; three (168 registers) spill and take 2.2 ms.
// SHARE: as for K (as a branch, (dd|dd) of 280 functions took 293 us, not 280).
template <int LA, int LB, int LC, int LD, typename G, bool SHARE>
__global__ __launch_bounds__(QX_RYS_BLOCK, sizeof(G) == 8 && qx_ncart(LC) * qx_ncart(LD) < 36 ? 2 : 1) void qx_rg(QxArgs A_, QxKList kl) {
  using S = QxRys<LA, LB, LC, LD, 1>;
  constexpr int NC = S::NC, ND = S::ND;
  HIP_DYNAMIC_SHARED(double, qx_sk)
  __shared__ double sg[QX_GRAD_LDS];
  G* const g = reinterpret_cast<G*>(qx_sk) + (threadIdx.x >> 6) * S::LDS;
  QxKBlock b;
  if (!qx_k_block(A_, kl, b)) return;
  const QxGradTarget tgt = qx_grad_begin(A_, kl, b.P1, sg);
  const QxRysLane<S, LA, LB> ln;
  const int n = A_.e.nbf, u1 = A_.pr.pp_first[b.P1];
  const double *da = A_.e.D + (size_t)(A_.pr.bfa[b.P1] + ln.ca) * n, *db = A_.e.D + (size_t)(A_.pr.bfb[b.P1] + ln.cb) * n;
  const double dab = ln.in ? da[A_.pr.bfb[b.P1] + ln.cb] : 0.0;
  G ab[3];
  {
    QxRysPair<G> bra;
    qx_rys_pair(A_, b.P1, u1, bra);
#pragma unroll
    for (int d = 0; d < 3; ++d) ab[d] = bra.AB[d];
  }
  double fi[3], fj[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    fi[d] = ln.e[d][0];
    fj[d] = ln.e[d][1];
  }
  double gb[6] = {}, gam[NC * ND];
  G v[9];
  bool act = false;
  int P2 = 0, pk = 0, nk = 0;
  qx_rys_walk<S, LB, LD, G, G, SHARE>(
      A_, kl, b, g,
      [&](int pk0, int nq) QX_INLINE {
        pk = pk0;
        nk = nq;
        const bool in = ln.in && ln.slot < nq;
        P2 = pk0 + (in ? ln.slot : 0);
        act = in && !qx_single_atom(A_, b.P1, P2);
        if (act) {
          const double f = 8.0 * qx_degeneracy(A_, b.P1, P2);
          const int ic = A_.pr.bfa[P2], id = A_.pr.bfb[P2];
          double ad[ND], bd[ND];
#pragma unroll
          for (int d = 0; d < ND; ++d) {
            ad[d] = 0.5 * f * da[id + d];
            bd[d] = 0.5 * f * db[id + d];
          }
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const double ac = da[ic + c], bc = db[ic + c];
            const double* dcd = A_.e.D + (size_t)(ic + c) * n + id;
#pragma unroll
            for (int d = 0; d < ND; ++d) gam[c * ND + d] = 2.0 * f * dab * dcd[d] - (ac * bd[d] + bc * ad[d]);
          }
        }
#pragma unroll
        for (int t = 0; t < 9; ++t) v[t] = G(0.0);
      },
      [&](int i1, int i2) QX_INLINE {
        if (!act || i2 >= A_.pr.pp_n[P2]) return;
        const double wa = A_.pp.a2[u1 + i1], wb = A_.pp.b2[u1 + i1], wc = A_.pp.a2[A_.pr.pp_first[P2] + i2];
        const G* gq = g + ln.slot * S::STRIDE;
#pragma unroll 1
        for (int r = 0; r < S::N; ++r) {
          const G* p[3];
          G o[3][S::NKU], w[3][S::NKU];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            p[x] = gq + (3 * r + x) * S::NG + ln.off(x);
#pragma unroll
            for (int k = 0; k < S::NKU; ++k) {
              o[x][k] = p[x][k];
              w[x][k] = G(0.0);
            }
          }
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int d = 0; d < ND; ++d) {
              const int kx = qx_comp(LC, c, 0) * (LD + 1) + qx_comp(LD, d, 0);
              const int ky = qx_comp(LC, c, 1) * (LD + 1) + qx_comp(LD, d, 1);
              const int kz = qx_comp(LC, c, 2) * (LD + 1) + qx_comp(LD, d, 2);
              const G gx = gam[c * ND + d] * o[0][kx], gz = gam[c * ND + d] * o[2][kz];
              w[0][kx] += o[1][ky] * gz;
              w[1][ky] += gx * o[2][kz];
              w[2][kz] += gx * o[1][ky];
            }
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            __builtin_amdgcn_sched_barrier(0);  // one direction's operands at a time in registers
            const G* up = p[x] + (LB + 1) * S::NKS;
            const G* dn = p[x] - (ln.e[x][0] > 0 ? (LB + 1) * S::NKS : 0);
            const G* bj = p[x] - (ln.e[x][1] > 0 ? S::NKS : 0);
            G su(0.0), sd(0.0), so(0.0), sb(0.0), sc(0.0), sk(0.0);
#pragma unroll
            for (int k = 0; k < S::NKU; ++k) {
              su += w[x][k] * up[k];
              sd += w[x][k] * dn[k];
              so += w[x][k] * o[x][k];
              sb += w[x][k] * bj[k];
              sc += w[x][k] * (k + LD + 1 < S::NKU ? o[x][k + LD + 1 < S::NKU ? k + LD + 1 : 0] : p[x][k + LD + 1]);
              if (k > LD) sk += (double(k / (LD + 1)) * w[x][k]) * o[x][k > LD ? k - LD - 1 : 0];
            }
            v[x] += wa * su - fi[x] * sd;
            v[3 + x] += wb * (su + ab[x] * so) - fj[x] * sb;
            v[6 + x] += wc * sc - sk;
          }
        }
      },
      [&]() QX_INLINE {
        // the ket centres' terms, summed over the quartet's lanes in LDS: one
        // LDS atomic per lane and direction would meet G-fold on each address
        // ((dd|ps) of 280 functions: 1.08 -> 0.79 ms)
        static_assert(6 * S::SUM * sizeof(double) <= S::LDS * sizeof(G), "LDS of the lane sums");
        double* const sum = reinterpret_cast<double*>(g);
        qx_wave_sync();
        if (ln.in) {
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const double a = act ? qx_value(v[x]) : 0.0, bb = act ? qx_value(v[3 + x]) : 0.0;
            const double c = act ? qx_value(v[6 + x]) : 0.0;
            gb[x] += a;
            gb[3 + x] += bb;
            sum[x * S::SUM + ln.slot * S::G + ln.ab] = c;
            sum[(3 + x) * S::SUM + ln.slot * S::G + ln.ab] = -(a + bb + c);
          }
        }
        qx_wave_sync();
        constexpr int PARTS = S::G % 3 == 0 ? 3 : 1, LEN = S::G / PARTS;
        for (int t = threadIdx.x & 63; t < nk * 6 * PARTS; t += 64) {
          const int q = t / (6 * PARTS), e = t - q * 6 * PARTS, x = e / PARTS, part = e - x * PARTS;
          const double* w = sum + x * S::SUM + q * S::G + part * LEN;
          double r = 0.0;
#pragma unroll
          for (int k = 0; k < LEN; ++k) r += w[k];
          tgt.add(3 * (x < 3 ? A_.pr.atom_a[pk + q] : A_.pr.atom_b[pk + q]) + (x < 3 ? x : x - 3), r);
        }
      });
  qx_grad_bra(A_, tgt, b.P1, gb);
  qx_grad_end(tgt);
}

// ---- launchers ----------------------------------------------------------------------
static inline dim3 qx_k_grid(const QxKList& kl) {
  return dim3((unsigned)kl.nbra, (unsigned)((kl.maxket + kl.chunk - 1) / kl.chunk), (unsigned)kl.psplit);
}

// K by quadrature (FP64 or FP32), and its directional derivative along tv.
#define QX_DEFINE_RYS_K_GO(NAME, LA, LB, LC, LD)                                                  \
  template <typename G, typename R>                                                               \
  static int qx_rk_go_##NAME(const QxArgs* a, const QxLaunch* L) {                                \
    using S = QxRys<LA, LB, LC, LD, 0>;                                                           \
    QxKList kl = *L->kl;                                                                          \
    const size_t W = a->e.kcols > 0 ? a->e.kcols : a->e.nbf, rows = (S::NA + S::NB) * W * sizeof(double);\
    const size_t wave = (size_t)S::LDS * sizeof(R);                                               \
    /* K' rows and density rows, else K' rows, else neither; eight wavefronts in one block where two\
       blocks of four do not fit */                                                               \
    int n = a->e.krows ? 2 : 0;                                                                   \
    while (n > 0 && n * rows + 4 * wave > QX_K_LDS_MAX) --n;                                      \
    const size_t base = n * rows;                                                                 \
    const int waves = 2 * (base + 4 * wave) > QX_K_LDS_MAX && base + 8 * wave <= QX_K_LDS_MAX ? 8 : 4;\
    const size_t sh = base + waves * wave;                                                        \
    /* values share primitives with both rows only: few workgroups means few functions */         \
    constexpr bool DUAL = sizeof(G) > sizeof(double);                                             \
    if (n < 2 && !DUAL) kl.psplit = 1;                                                            \
    auto kernel = n == 1 ? qx_rk<LA, LB, LC, LD, G, R, true, false, DUAL> : qx_rk<LA, LB, LC, LD, G, R, false, false, DUAL>;\
    if (n == 2) kernel = kl.psplit > 1 ? qx_rk<LA, LB, LC, LD, G, R, true, true, true> : qx_rk<LA, LB, LC, LD, G, R, true, true, DUAL>;\
    hipLaunchKernelGGL(kernel, qx_k_grid(kl), dim3(64 * waves), sh, L->stream, *a, kl);           \
    return (int)hipGetLastError();                                                                \
  }
#define QX_DEFINE_RYS_K(NAME, LA, LB, LC, LD, WITH32)                                             \
  QX_DEFINE_RYS_K_GO(NAME, LA, LB, LC, LD)                                                        \
  extern "C" int qx_launchj_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    if (L->fp32 == 0) return qx_rk_go_##NAME<double, double>(a, L);                               \
    if constexpr (WITH32) {                                                                       \
      if (L->fp32 == 1) return qx_rk_go_##NAME<double, float>(a, L);                              \
    }                                                                                             \
    return -1;                                                                                    \
  }

#define QX_DEFINE_RYS_KV(NAME, LA, LB, LC, LD)                                                    \
  QX_DEFINE_RYS_K_GO(v##NAME, LA, LB, LC, LD)                                                     \
  extern "C" int qx_launchv_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    return a->e.tv ? qx_rk_go_v##NAME<qx_dual, qx_dual>(a, L) : -1;                               \
  }

// Integrals (QX_DEFINE_RYS_E: pair matrix, store, Schwarz) and derivative integrals (QX_DEFINE_RYS_D, with
// L->fp32 = 2 their derivatives along tv) into the pair matrix.
#define QX_DEFINE_RYS_E(NAME, LA, LB, LC, LD)                                                     \
  extern "C" int qx_launch_##NAME(const QxArgs* a, const QxLaunch* L) {                           \
    if (!L->kl || L->fp32 || a->e.epi == QX_EPI_JK) return -1;                                    \
    if constexpr (LA == LC && LB == LD) {                                                         \
      if (a->e.epi == QX_EPI_SCHWARZ) {                                                           \
        if (L->kl->nbra <= 0) return 0;                                                           \
        const size_t one = sizeof(double) * QxRys<LA, LB, LA, LB, 0>::LDS;                        \
        hipLaunchKernelGGL((qx_rs<LA, LB>), dim3((unsigned)L->kl->nbra), dim3(64), one, L->stream, *a, *L->kl); \
        return (int)hipGetLastError();                                                            \
      }                                                                                           \
    }                                                                                             \
    if (L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                                       \
    const bool store = a->e.epi == QX_EPI_STORE;                                                  \
    if (store ? L->kl->ketprim != 1 : !L->pm) return -1;                                          \
    const size_t sh = 4 * sizeof(double) * QxRys<LA, LB, LC, LD, 0>::LDS;                         \
    auto kernel = store ? qx_re<LA, LB, LC, LD, 2> : L->kl->psplit > 1 ? qx_re<LA, LB, LC, LD, 1> : qx_re<LA, LB, LC, LD, 0>; \
    hipLaunchKernelGGL(kernel, qx_k_grid(*L->kl), dim3(QX_RYS_BLOCK), sh, L->stream, *a, *L->kl, \
                       store ? QxPairM{} : *L->pm);                                               \
    return (int)hipGetLastError();                                                                \
  }
#define QX_DEFINE_RYS_D(NAME, LA, LB, LC, LD)                                                     \
  extern "C" int qx_launch_##NAME(const QxArgs* a, const QxLaunch* L) {                           \
    if (!L->kl || !L->pm || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                   \
    const size_t values = 4 * (size_t)QxRys<LA, LB, LC, LD, 1>::LDS;                              \
    if (L->fp32 == 0)                                                                             \
      hipLaunchKernelGGL((qx_rd<LA, LB, LC, LD, double>), qx_k_grid(*L->kl), dim3(QX_RYS_BLOCK), values * sizeof(double), \
                         L->stream, *a, *L->kl, *L->pm);                                          \
    else if (L->fp32 == 2)                                                                        \
      hipLaunchKernelGGL((qx_rd<LA, LB, LC, LD, qx_dual>), qx_k_grid(*L->kl), dim3(QX_RYS_BLOCK), values * sizeof(qx_dual), \
                         L->stream, *a, *L->kl, *L->pm);                                          \
    else return -1;                                                                               \
    return (int)hipGetLastError();                                                                \
  }

// Adjoint gradient (in FP64 also where a mixed pass asks for FP32), and its
// derivative along tv.
template <int LA, int LB, int LC, int LD, typename G>
static int qx_rg_go(const QxArgs* a, const QxLaunch* L) {
  const size_t sh = 4 * (size_t)QxRys<LA, LB, LC, LD, 1>::LDS * sizeof(G);
  constexpr bool DUAL = sizeof(G) > sizeof(double);
  auto kernel = L->kl->psplit > 1 ? qx_rg<LA, LB, LC, LD, G, true> : qx_rg<LA, LB, LC, LD, G, DUAL>;
  hipLaunchKernelGGL(kernel, qx_k_grid(*L->kl), dim3(QX_RYS_BLOCK), sh, L->stream, *a, *L->kl);
  return (int)hipGetLastError();
}
#define QX_DEFINE_RYS_G(NAME, LA, LB, LC, LD)                                                     \
  extern "C" int qx_launchg_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    return qx_rg_go<LA, LB, LC, LD, double>(a, L);                                                \
  }
#define QX_DEFINE_RYS_H(NAME, LA, LB, LC, LD)                                                     \
  extern "C" int qx_launchh_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    return a->e.tv ? qx_rg_go<LA, LB, LC, LD, qx_dual>(a, L) : -1;                       \
  }
