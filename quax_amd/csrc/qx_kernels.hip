// Helper kernels of the ERI library: fills, symmetrisation, Cartesian <->
// spherical transforms, and the one-electron integrals (overlap, kinetic,
// nuclear attraction) with their first nuclear derivatives.
//
// One-electron integrals are O(n^2 N) work next to the O(n^4) two-electron
// path, so these kernels favour compact generic code: one thread per ordered
// shell pair, 1D Obara-Saika tables for S and T, an Obara-Saika vertical
// recurrence on the bra for V followed by the binomial transfer
// (a|O|b) = sum_k C(b,k) AB^(b-k) (a+k|O|0) per Cartesian direction.
#include <hip/hip_runtime.h>

#include "qx_runtime.h"

namespace {

// 16-byte stores where p allows, a few per lane: the 0.43 GB pair matrix of a
// 112-function tensor takes 0.08 ms (8-byte stores, one per lane: 0.39 ms).
__global__ __launch_bounds__(256) void k_fill(double* p, long long n, double v) {
  const long long step = (long long)gridDim.x * blockDim.x, i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if ((reinterpret_cast<size_t>(p) & 15) == 0) {
    double2* q = reinterpret_cast<double2*>(p);
    for (long long i = i0; i < n / 2; i += step) q[i] = make_double2(v, v);
    if (i0 == 0 && (n & 1)) p[n - 1] = v;
  } else {
    for (long long i = i0; i < n; i += step) p[i] = v;
  }
}

// out[i] += sum_c copies[c * n + i]
__global__ void k_add_copies(const double* copies, int ncopy, int n, double* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = 0.0;
  for (int c = 0; c < ncopy; ++c) v += copies[(size_t)c * n + i];
  out[i] += v;
}

// AO function k of shell s: row of the transform block; Cartesian function p
// of the same shell: column.
__device__ __forceinline__ double tcoef(const QxShellsDev& sh, int s, int row, int col) {
  const int l = sh.l[s];
  const int nc = (l + 1) * (l + 2) / 2;
  return sh.sph[sh.sph_off[l] + row * nc + col];
}

// out[i][j] = sum_{p in shell(i), q in shell(j)} T[i][p] X[p][q] T[j][q]
__device__ __forceinline__ void cart_to_ao_at(const QxShellsDev& sh, const double* X, double* out) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = sh.nbf, nc = sh.ncart;
  if (t >= (long long)nb * nb) return;
  const int i = (int)(t / nb), j = (int)(t % nb);
  const int si = sh.ao_shell[i], sj = sh.ao_shell[j];
  const int ri = i - sh.bfs[si], rj = j - sh.bfs[sj];
  const int li = sh.l[si], lj = sh.l[sj];
  const int ni = (li + 1) * (li + 2) / 2, nj = (lj + 1) * (lj + 2) / 2;
  double acc = 0.0;
  for (int p = 0; p < ni; ++p) {
    const double tp = tcoef(sh, si, ri, p);
    if (tp == 0.0) continue;
    for (int q = 0; q < nj; ++q) acc += tp * X[(size_t)(sh.bfc[si] + p) * nc + sh.bfc[sj] + q] * tcoef(sh, sj, rj, q);
  }
  out[t] = acc;
}

// out[p][q] = sum_{i in shell(p), j in shell(q)} T[i][p] X[i][j] T[j][q]
__device__ __forceinline__ void ao_to_cart_at(const QxShellsDev& sh, const double* X, double* out) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = sh.nbf, nc = sh.ncart;
  if (t >= (long long)nc * nc) return;
  const int p = (int)(t / nc), q = (int)(t % nc);
  const int sp = sh.f_shell[p], sq = sh.f_shell[q];
  const int cp = p - sh.bfc[sp], cq = q - sh.bfc[sq];
  const int np = (sh.pure && sh.l[sp] >= 2) ? 2 * sh.l[sp] + 1 : (sh.l[sp] + 1) * (sh.l[sp] + 2) / 2;
  const int nq = (sh.pure && sh.l[sq] >= 2) ? 2 * sh.l[sq] + 1 : (sh.l[sq] + 1) * (sh.l[sq] + 2) / 2;
  double acc = 0.0;
  for (int i = 0; i < np; ++i) {
    const double ti = tcoef(sh, sp, i, cp);
    if (ti == 0.0) continue;
    for (int j = 0; j < nq; ++j) acc += ti * X[(size_t)(sh.bfs[sp] + i) * nb + sh.bfs[sq] + j] * tcoef(sh, sq, j, cq);
  }
  out[t] = acc;
}

// Up to three matrices at once (grid row y): the kernels' arithmetic is that of
// the single forms above.
struct MatPtrs {
  const double* in[3];
  double* out[3];
};
__global__ void k_cart_to_ao_mats(QxShellsDev sh, MatPtrs m) { cart_to_ao_at(sh, m.in[blockIdx.y], m.out[blockIdx.y]); }
__global__ void k_ao_to_cart_mats(QxShellsDev sh, MatPtrs m) { ao_to_cart_at(sh, m.in[blockIdx.y], m.out[blockIdx.y]); }

// ---------------------------------------------------------------- pair matrix
__global__ void k_fill_int(int* p, long long n, int v) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// One thread per screened shell pair: its function pairs' rows.
__global__ void k_pairm_index(QxShellsDev sh, QxPairsDev pr, int npairs, QxPairIndex ix, int* index, int* fn) {
  const int P = blockIdx.x * blockDim.x + threadIdx.x;
  if (P >= npairs) return;
  const int la = sh.l[pr.sa[P]], lb = sh.l[pr.sb[P]];
  const int na = (la + 1) * (la + 2) / 2, nb = (lb + 1) * (lb + 2) / 2, n = sh.ncart;
  int X = la * (la + 1) / 2 + lb, off = 0;
  for (int k = 0; k < X; ++k) off += ix.cnt[k];
  const bool diag = pr.sa[P] == pr.sb[P];  // both orders are components of the block
  for (int i = 0; i < na; ++i)
    for (int j = 0; j < nb; ++j) {
      const int row = ix.base[X] + (i * nb + j) * ix.cnt[X] + (P - off);
      index[(size_t)(pr.bfa[P] + i) * n + pr.bfb[P] + j] = row;
      fn[row] = (pr.bfa[P] + i) * n + pr.bfb[P] + j;
      if (!diag) index[(size_t)(pr.bfb[P] + j) * n + pr.bfa[P] + i] = row;
    }
}

// One thread per AO function: its Cartesian terms.
__global__ void k_ao_terms(QxShellsDev sh, QxAoTerms* ao) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= sh.nbf) return;
  const int s = sh.ao_shell[r], l = sh.l[s], nc = (l + 1) * (l + 2) / 2;
  QxAoTerms t{};
  for (int p = 0; p < nc; ++p) {
    const double c = tcoef(sh, s, r - sh.bfs[s], p);
    if (c == 0.0 || t.n == 3) continue;
    t.f[t.n] = sh.bfc[s] + p;
    t.c[t.n++] = c;
  }
  ao[r] = t;
}

// Class and pair position of row r.
__device__ __forceinline__ void pairm_row(const QxPairIndex& ix, int r, int& X, int& pos) {
  X = 0;
#pragma unroll
  for (int k = 1; k < 6; ++k) X = r >= ix.base[k] ? k : X;
  pos = (r - ix.base[X]) % max(ix.cnt[X], 1);
}

// The quartet kernels store (row, column) for bra class > ket class, or bra
// position >= ket position within a class; the other elements are the
// transposed ones.  A workgroup owns the 64 x 64 tile (tr, tc) and its mirror
// image, so it reads both before it writes either.  Bound by HBM: half of M
// read and written.
#define PM_TILE 64
#define PM_LDS_MAX (140 * 1024)  // a staged row; the rest of a workgroup's 160 KB holds the term lists
#define PM_AO_MAX 384            // AO functions whose term lists are kept in LDS
__global__ __launch_bounds__(256) void k_pairm_sym(double* M, long long ld, long long slice, QxPairIndex ix) {
  __shared__ double a[PM_TILE][PM_TILE + 1], b[PM_TILE][PM_TILE + 1];
  M += (long long)blockIdx.y * slice;
  const long long t = blockIdx.x;
  int tr = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(tr + 1) * (tr + 2) / 2 <= t) ++tr;
  while ((long long)tr * (tr + 1) / 2 > t) --tr;
  const int tc = (int)(t - (long long)tr * (tr + 1) / 2);
  const int r0 = tr * PM_TILE, c0 = tc * PM_TILE;
  const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
  for (int y = ly; y < PM_TILE; y += 4) {
    a[y][lx] = r0 + y < ld && c0 + lx < ld ? M[(long long)(r0 + y) * ld + c0 + lx] : 0.0;
    b[y][lx] = c0 + y < ld && r0 + lx < ld ? M[(long long)(c0 + y) * ld + r0 + lx] : 0.0;
  }
  __syncthreads();
  for (int y = ly; y < PM_TILE; y += 4) {
    int Xr, Xc, pr, pc;
    if (r0 + y < ld && c0 + lx < ld) {          // element (r0 + y, c0 + lx)
      pairm_row(ix, r0 + y, Xr, pr);
      pairm_row(ix, c0 + lx, Xc, pc);
      const bool there = Xr > Xc || (Xr == Xc && pr >= pc);
      if (!there) M[(long long)(r0 + y) * ld + c0 + lx] = b[lx][y];
    }
    if (c0 + y < ld && r0 + lx < ld && tr != tc) {  // element (c0 + y, r0 + lx)
      pairm_row(ix, c0 + y, Xr, pr);
      pairm_row(ix, r0 + lx, Xc, pc);
      const bool there = Xr > Xc || (Xr == Xc && pr >= pc);
      if (!there) M[(long long)(c0 + y) * ld + r0 + lx] = a[lx][y];
    }
  }
}

// The elements of a panel of rows (pairs [i0, i0 + cnt) of class X, ncomp
// components) to all their places in a Cartesian tensor: eight scattered
// stores per element, used only when no whole pair matrix fits in memory.
__global__ void k_pairm_scatter(int nc, const double* M, long long ld, long long slice, QxPairIndex ix, const int* fn,
                                int X, int ncomp, int i0, int cnt, double* out) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int rows = ncomp * cnt, cols = ix.base[X + 1];  // kets of class X and below
  if (t >= (long long)rows * cols) return;
  const int pr = (int)(t / cols), col = (int)(t - (long long)pr * cols);
  int Y, j;
  pairm_row(ix, col, Y, j);
  const int k = pr / cnt, i = i0 + (pr - k * cnt);
  if (Y > X || (Y == X && j > i)) return;
  const double v = M[(long long)blockIdx.y * slice + (long long)pr * ld + col];
  const int pq = fn[ix.base[X] + k * ix.cnt[X] + i], rs = fn[col];
  const size_t n = nc, p = pq / nc, q = pq % nc, r = rs / nc, u = rs % nc;
  double* o = out + (size_t)blockIdx.y * n * n * n * n;
  o[((p * n + q) * n + r) * n + u] = v;
  o[((q * n + p) * n + r) * n + u] = v;
  o[((p * n + q) * n + u) * n + r] = v;
  o[((q * n + p) * n + u) * n + r] = v;
  o[((r * n + u) * n + p) * n + q] = v;
  o[((u * n + r) * n + p) * n + q] = v;
  o[((r * n + u) * n + q) * n + p] = v;
  o[((u * n + r) * n + q) * n + p] = v;
}

// One workgroup per AO function pair p >= q (and slice): the row of (p, q),
// transformed to AO on its two bra indices, is staged in LDS (or read in
// place when it does not fit, STAGE = false), then written to out[p][q] and
// out[q][p] with the ket transform applied: consecutive lanes write
// consecutive doubles.  Bound by the tensor's HBM writes.
template <bool PURE, bool STAGE>
__global__ __launch_bounds__(256) void k_pairm_expand(int n, int nc, const double* M, long long ld, long long slice,
                                                      const int* index, const QxAoTerms* ao, double* out) {
  HIP_DYNAMIC_SHARED(double, row)
  __shared__ QxAoTerms terms[PURE ? PM_AO_MAX : 1];  // AO terms, where they fit
  __shared__ long long src[9];
  __shared__ double coef[9];
  __shared__ int nsrc;
  const long long t = blockIdx.x;
  int p = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(p + 1) * (p + 2) / 2 <= t) ++p;
  while ((long long)p * (p + 1) / 2 > t) --p;
  const int q = (int)(t - (long long)p * (p + 1) / 2);
  M += (long long)blockIdx.y * slice;
  if (threadIdx.x == 0) {
    int k = 0;
    if (PURE) {
      const QxAoTerms tp = ao[p], tq = ao[q];
      for (int i = 0; i < tp.n; ++i)
        for (int j = 0; j < tq.n; ++j) {
          const int r = index[(size_t)tp.f[i] * nc + tq.f[j]];
          if (r >= 0) { src[k] = r * ld; coef[k++] = tp.c[i] * tq.c[j]; }
        }
    } else {
      const int r = index[(size_t)p * nc + q];
      if (r >= 0) { src[k] = r * ld; coef[k++] = 1.0; }
    }
    nsrc = k;
  }
  const bool near = PURE && n <= PM_AO_MAX;
  if (near)
    for (int i = threadIdx.x; i < n; i += blockDim.x) terms[i] = ao[i];
  __syncthreads();
  const int ns = nsrc;
  if (STAGE) {
    for (int c = threadIdx.x; c < ld; c += blockDim.x) {
      double v = 0.0;
      for (int k = 0; k < ns; ++k) v += coef[k] * M[src[k] + c];
      row[c] = v;
    }
    __syncthreads();
  }
  auto at = [&](int c) -> double {
    if (c < 0) return 0.0;
    if (STAGE) return row[c];
    double v = 0.0;
    for (int k = 0; k < ns; ++k) v += coef[k] * M[src[k] + c];
    return v;
  };
  const long long nn = (long long)n * n;
  double* o1 = out + (long long)blockIdx.y * nn * nn + ((long long)p * n + q) * nn;
  double* o2 = out + (long long)blockIdx.y * nn * nn + ((long long)q * n + p) * nn;
  for (int i = threadIdx.x; i < nn; i += blockDim.x) {
    double v;
    if (PURE) {
      const int r = i / n, u = i - r * n;
      const QxAoTerms* tr = near ? &terms[r] : ao + r;
      const QxAoTerms* tu = near ? &terms[u] : ao + u;
      const int nr = tr->n, nu = tu->n;
      v = 0.0;
      for (int x = 0; x < nr; ++x) {
        const int* ix = index + (size_t)tr->f[x] * nc;
        const double cx = tr->c[x];
        for (int y = 0; y < nu; ++y) v += cx * tu->c[y] * at(ix[tu->f[y]]);
      }
    } else {
      v = at(index[i]);
    }
    o1[i] = v;
    if (p != q) o2[i] = v;
  }
}

// ---------------------------------------------------------------- OEI
#define OE_LMAX 3          // bra/ket l after a derivative shift
#define OE_JMAX (OE_LMAX + 2)
#define OE_LT (2 * OE_LMAX)

__device__ __forceinline__ int d_coff(int l) { return l * (l + 1) * (l + 2) / 6; }
__device__ __forceinline__ int d_gidx(int x, int y, int z) {
  const int i = y + z;
  return d_coff(x + y + z) + i * (i + 1) / 2 + z;
}

__device__ void oe_boys(int M, double T, double* F) {
  // direct series / asymptotic evaluation (one-electron integrals only)
  if (T < 35.0) {
    double term = 1.0 / (2 * M + 1), sum = term;
    for (int k = 1; k < 300; ++k) {
      term *= 2.0 * T / (2 * M + 2 * k + 1);
      sum += term;
      if (term < 1e-17 * sum) break;
    }
    const double et = exp(-T);
    F[M] = et * sum;
    for (int m = M; m > 0; --m) F[m - 1] = (2.0 * T * F[m] + et) / (2 * m - 1);
  } else {
    const double et = exp(-T);
    F[0] = 0.5 * sqrt(3.14159265358979323846 / T);
    for (int m = 0; m < M; ++m) F[m + 1] = ((2 * m + 1) * F[m] - et) / (2.0 * T);
  }
}

struct OePrim {
  double a, b, p;      // exponents, p = a+b
  double K;            // ca cb exp(-ab/p AB^2)
  double PA[3], PB[3], AB[3];
};

// 1D overlap tables s[d][i][j] (no prefactor), i <= imax, j <= jmax
__device__ void oe_s1d(const OePrim& P, int imax, int jmax, double (*s)[OE_LMAX + 2][OE_JMAX + 2]) {
  const double o2p = 0.5 / P.p;
  for (int d = 0; d < 3; ++d)
    for (int j = 0; j <= jmax; ++j)
      for (int i = 0; i <= imax; ++i) {
        double v;
        if (i == 0 && j == 0) v = 1.0;
        else if (j == 0) {
          v = P.PA[d] * s[d][i - 1][0];
          if (i > 1) v += o2p * (i - 1) * s[d][i - 2][0];
        } else {
          v = P.PB[d] * s[d][i][j - 1];
          if (i > 0) v += o2p * i * s[d][i - 1][j - 1];
          if (j > 1) v += o2p * (j - 1) * s[d][i][j - 2];
        }
        s[d][i][j] = v;
      }
}

// S and T for component pair (a, b) from the 1D tables
__device__ __forceinline__ void oe_st(const OePrim& P, const int* a, const int* b,
                                      double (*s)[OE_LMAX + 2][OE_JMAX + 2], double& Sv, double& T) {
  const double pref = pow(3.14159265358979323846 / P.p, 1.5);
  double sv[3], tv[3];
  for (int d = 0; d < 3; ++d) {
    const int i = a[d], j = b[d];
    sv[d] = s[d][i][j];
    double t = P.b * (2 * j + 1) * s[d][i][j] - 2.0 * P.b * P.b * s[d][i][j + 2];
    if (j > 1) t = t - 0.5 * j * (j - 1) * s[d][i][j - 2];
    tv[d] = t;
  }
  Sv = pref * sv[0] * sv[1] * sv[2];
  T = pref * (tv[0] * sv[1] * sv[2] + sv[0] * tv[1] * sv[2] + sv[0] * sv[1] * tv[2]);
}

// [e|0]^(0) for |e| <= L toward a unit charge at C (no -Z, includes 2pi/p K)
__device__ void oe_vrr(const OePrim& P, const double* Pc, const double* C, int L, double* out /*coff(L+1)*/) {
  double V[OE_LT + 1][56];
  double PC[3] = {Pc[0] - C[0], Pc[1] - C[1], Pc[2] - C[2]};
  const double T = P.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]);
  double F[OE_LT + 2];
  oe_boys(L, T, F);
  const double pref = 2.0 * 3.14159265358979323846 / P.p * P.K;
  for (int m = 0; m <= L; ++m) V[m][0] = pref * F[m];
  const double o2p = 0.5 / P.p;
  for (int l = 1; l <= L; ++l)
    for (int i = 0; i <= l; ++i)
      for (int j = 0; j <= i; ++j) {
        const int e[3] = {l - i, i - j, j};
        const int ax = e[0] > 0 ? 0 : (e[1] > 0 ? 1 : 2);
        int e1[3] = {e[0], e[1], e[2]};
        e1[ax] -= 1;
        const int g = d_gidx(e[0], e[1], e[2]), g1 = d_gidx(e1[0], e1[1], e1[2]);
        int g2 = -1;
        if (e1[ax] > 0) {
          int e2[3] = {e1[0], e1[1], e1[2]};
          e2[ax] -= 1;
          g2 = d_gidx(e2[0], e2[1], e2[2]);
        }
        for (int m = 0; m <= L - l; ++m) {
          double v = P.PA[ax] * V[m][g1] - PC[ax] * V[m + 1][g1];
          if (g2 >= 0) v = v + o2p * e1[ax] * (V[m][g2] - V[m + 1][g2]);
          V[m][g] = v;
        }
      }
  for (int g = 0; g < d_coff(L + 1); ++g) out[g] = V[0][g];
}

__device__ __forceinline__ double binom(int n, int k) {
  double r = 1.0;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}

// (a|V_C|b) from the [e|0] table by the binomial transfer
__device__ double oe_vab(const double* E, const int* a, const int* b, const double* AB) {
  double acc = 0.0;
  for (int kx = 0; kx <= b[0]; ++kx)
    for (int ky = 0; ky <= b[1]; ++ky)
      for (int kz = 0; kz <= b[2]; ++kz) {
        const double c = binom(b[0], kx) * binom(b[1], ky) * binom(b[2], kz) * pow(AB[0], b[0] - kx) *
                         pow(AB[1], b[1] - ky) * pow(AB[2], b[2] - kz);
        acc = acc + c * E[d_gidx(a[0] + kx, a[1] + ky, a[2] + kz)];
      }
  return acc;
}

__device__ void unpack(int code, int* c) {
  c[0] = code >> 16;
  c[1] = (code >> 8) & 0xff;
  c[2] = code & 0xff;
}

__device__ OePrim oe_prim(const QxShellsDev& sh, int sa, int sb, int ia, int ib) {
  OePrim P;
  const double *A = sh.xyz + 3 * sh.atom[sa], *B = sh.xyz + 3 * sh.atom[sb];
  P.a = sh.exps[ia];
  P.b = sh.exps[ib];
  P.p = P.a + P.b;
  double AB2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double Pd = (P.a * A[d] + P.b * B[d]) / P.p;
    P.PA[d] = Pd - A[d];
    P.PB[d] = Pd - B[d];
    P.AB[d] = A[d] - B[d];
    AB2 += P.AB[d] * P.AB[d];
  }
  P.K = sh.coefs[ia] * sh.coefs[ib] * exp(-P.a * P.b / P.p * AB2);
  return P;
}

// Derivative tensors dS, dT, dV (3N x n x n, accumulated): d/dA_x of (a|O|b) =
// 2 alpha (a+1_x|O|b) - a_x (a-1_x|O|b), same on b; the nuclear-attraction
// operator centre follows from translational invariance of each nucleus term.
// Thread x takes one ordered shell pair; grid row y takes the terms: 0 the
// overlap and kinetic ones, 1 + C the attraction of nucleus C (rows stride by
// gridDim.y), so a pair's nucleus loop is spread over the grid instead of run
// by one lane.
__global__ void k_oei_deriv(QxShellsDev sh, double* dS, double* dT, double* dV) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= sh.nshell * sh.nshell) return;
  const int sa = t / sh.nshell, sb = t % sh.nshell;
  const int la = sh.l[sa], lb = sh.l[sb];
  const int na = (la + 1) * (la + 2) / 2, nb = (lb + 1) * (lb + 2) / 2;
  const int n = sh.ncart;
  const size_t nn = (size_t)n * n;
  const int atA = sh.atom[sa], atB = sh.atom[sb];
  double s1[3][OE_LMAX + 2][OE_JMAX + 2];
  double E[84];
  for (int term = blockIdx.y; term <= sh.natom; term += gridDim.y) {
    for (int ia = sh.poff[sa]; ia < sh.poff[sa] + sh.nprim[sa]; ++ia)
      for (int ib = sh.poff[sb]; ib < sh.poff[sb] + sh.nprim[sb]; ++ib) {
        const OePrim P = oe_prim(sh, sa, sb, ia, ib);
        const int atC = term - 1;
        if (term == 0) {
          oe_s1d(P, la + 1, lb + 3, s1);
        } else {
          double Pc[3];
          for (int d = 0; d < 3; ++d) Pc[d] = sh.xyz[3 * atA + d] + P.PA[d];
          oe_vrr(P, Pc, sh.xyz + 3 * atC, la + lb + 1, E);
        }
        for (int i = 0; i < na; ++i)
          for (int j = 0; j < nb; ++j) {
            int a[3], b[3];
            unpack(sh.f_comp[sh.bfc[sa] + i], a);
            unpack(sh.f_comp[sh.bfc[sb] + j], b);
            const size_t rc = (size_t)(sh.bfc[sa] + i) * n + sh.bfc[sb] + j;
            for (int side = 0; side < 2; ++side) {
              const double ex2 = 2.0 * (side == 0 ? P.a : P.b);
              const int at = side == 0 ? atA : atB;
              for (int x = 0; x < 3; ++x) {
                int au[3] = {a[0], a[1], a[2]}, bu[3] = {b[0], b[1], b[2]};
                if (side == 0) au[x] += 1; else bu[x] += 1;
                const int q = side == 0 ? a[x] : b[x];
                int ad[3] = {a[0], a[1], a[2]}, bd[3] = {b[0], b[1], b[2]};
                if (side == 0) ad[x] -= 1; else bd[x] -= 1;
                if (term == 0) {  // overlap and kinetic
                  double su, tu, ds, dt;
                  oe_st(P, au, bu, s1, su, tu);
                  ds = ex2 * su;
                  dt = ex2 * tu;
                  if (q > 0) {
                    double sd, td;
                    oe_st(P, ad, bd, s1, sd, td);
                    ds -= q * sd;
                    dt -= q * td;
                  }
                  atomicAdd(&dS[(size_t)(3 * at + x) * nn + rc], P.K * ds);
                  atomicAdd(&dT[(size_t)(3 * at + x) * nn + rc], P.K * dt);
                  continue;
                }
                double dv = ex2 * oe_vab(E, au, bu, P.AB);
                if (q > 0) dv -= q * oe_vab(E, ad, bd, P.AB);
                dv *= -sh.Z[atC];
                atomicAdd(&dV[(size_t)(3 * at + x) * nn + rc], dv);
                atomicAdd(&dV[(size_t)(3 * atC + x) * nn + rc], -dv);
              }
            }
          }
      }
  }
}

inline unsigned nblk(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

extern "C" {

int qxk_fill(double* p, long long n, double v, hipStream_t s) {
  if (n <= 0) return 0;
  const long long blocks = std::min<long long>((n + 511) / 512, 8192);
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  return (int)hipGetLastError();
}

int qxk_add_copies(const double* copies, int ncopy, int n, double* out, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_add_copies, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, copies, ncopy, n, out);
  return (int)hipGetLastError();
}

int qxk_cart_to_ao_mats(const QxShellsDev* sh, const double* in, size_t stride, double* const* out, int count,
                        hipStream_t s) {
  MatPtrs m{};
  for (int k = 0; k < count; ++k) { m.in[k] = in + k * stride; m.out[k] = out[k]; }
  hipLaunchKernelGGL(k_cart_to_ao_mats, dim3(nblk((long long)sh->nbf * sh->nbf, 256), (unsigned)count), dim3(256), 0, s,
                     *sh, m);
  return (int)hipGetLastError();
}

int qxk_ao_to_cart_mats(const QxShellsDev* sh, const double* const* in, double* out, size_t stride, int count,
                        hipStream_t s) {
  MatPtrs m{};
  for (int k = 0; k < count; ++k) { m.in[k] = in[k]; m.out[k] = out + k * stride; }
  hipLaunchKernelGGL(k_ao_to_cart_mats, dim3(nblk((long long)sh->ncart * sh->ncart, 256), (unsigned)count), dim3(256), 0,
                     s, *sh, m);
  return (int)hipGetLastError();
}

int qxk_cart_to_ao_mat(const QxShellsDev* sh, const double* in, double* out, hipStream_t s) {
  return qxk_cart_to_ao_mats(sh, in, 0, &out, 1, s);
}

int qxk_ao_to_cart_mat(const QxShellsDev* sh, const double* in, double* out, hipStream_t s) {
  return qxk_ao_to_cart_mats(sh, &in, out, 0, 1, s);
}

int qxk_pairm_tables(const QxShellsDev* sh, const QxPairsDev* pr, int npairs, const QxPairIndex* ix, int* index,
                     int* fn, QxAoTerms* ao, hipStream_t s) {
  const long long n2 = (long long)sh->ncart * sh->ncart;
  hipLaunchKernelGGL(k_fill_int, dim3(std::min(nblk(n2, 256), 4096u)), dim3(256), 0, s, index, n2, -1);
  if (npairs > 0)
    hipLaunchKernelGGL(k_pairm_index, dim3(nblk(npairs, 128)), dim3(128), 0, s, *sh, *pr, npairs, *ix, index, fn);
  if (sh->pure) hipLaunchKernelGGL(k_ao_terms, dim3(nblk(sh->nbf, 128)), dim3(128), 0, s, *sh, ao);
  return (int)hipGetLastError();
}

int qxk_pairm_sym(double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix, hipStream_t s) {
  const long long T = (ld + PM_TILE - 1) / PM_TILE, tiles = T * (T + 1) / 2;
  if (tiles <= 0 || nslice <= 0) return 0;
  if (tiles > 0x7fffffffLL || nslice > 65535) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pairm_sym, dim3((unsigned)tiles, (unsigned)nslice), dim3(256), 0, s, M, ld, slice, *ix);
  return (int)hipGetLastError();
}

int qxk_pairm_scatter(int ncart, const double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix,
                      const int* fn, int X, int ncomp, int i0, int cnt, double* out, hipStream_t s) {
  const long long total = (long long)ncomp * cnt * ix->base[X + 1];
  if (total <= 0 || nslice <= 0) return 0;
  if ((total + 255) / 256 > 0x7fffffffLL || nslice > 65535) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pairm_scatter, dim3(nblk(total, 256), (unsigned)nslice), dim3(256), 0, s, ncart, M, ld, slice,
                     *ix, fn, X, ncomp, i0, cnt, out);
  return (int)hipGetLastError();
}

int qxk_pairm_expand(const QxShellsDev* sh, const double* M, long long ld, long long slice, int nslice,
                     const int* index, const QxAoTerms* ao, double* out, hipStream_t s) {
  const int n = sh->nbf;
  const dim3 grid((unsigned)((long long)n * (n + 1) / 2), (unsigned)nslice);
  if (nslice <= 0) return 0;
  if (nslice > 65535) return (int)hipErrorInvalidValue;
  const size_t bytes = (size_t)ld * sizeof(double);
  const bool stage = bytes <= PM_LDS_MAX;
#define PM_GO(P, S) hipLaunchKernelGGL((k_pairm_expand<P, S>), grid, dim3(256), (S) ? bytes : 0, s, n, sh->ncart, M, ld, slice, index, ao, out)
  if (sh->pure) { if (stage) PM_GO(true, true); else PM_GO(true, false); }
  else { if (stage) PM_GO(false, true); else PM_GO(false, false); }
#undef PM_GO
  return (int)hipGetLastError();
}

int qxk_oei_deriv(const QxShellsDev* sh, double* dS, double* dT, double* dV, hipStream_t s) {
  const unsigned rows = (unsigned)std::min(sh->natom + 1, 65535);
  hipLaunchKernelGGL(k_oei_deriv, dim3(nblk((long long)sh->nshell * sh->nshell, 64), rows), dim3(64), 0, s, *sh, dS, dT,
                     dV);
  return (int)hipGetLastError();
}

}  // extern "C"
