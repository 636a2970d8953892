// Helper kernels of the ERI library: fills, Cartesian <-> spherical transforms,
// the pair matrix's way to a tensor, and the derivative matrices of the
// one-electron integrals (their values and contracted derivatives: qx_oei.h).
//
// The derivative matrices are O(n^2 N) work next to the O(n^4) two-electron
// path, so their kernel favours compact generic code: one thread per ordered
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

// Up to three matrices at once (grid row y).
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

// Screened shell pair P: the rows of its AO function pairs (index) and the
// function pair of each row (fn: higher << 16 | lower, -1 for a component no
// pair has).  A pair's AO components take the first of the rows its Cartesian
// ones had.
__device__ __forceinline__ void pairm_index(const QxShellsDev& sh, const QxPairsDev& pr, int P, const QxPairIndex& ix,
                                            int* index, int* fn) {
  const int la = sh.l[pr.sa[P]], lb = sh.l[pr.sb[P]], n = sh.nbf;
  const int na = sh.pure && la > 1 ? 2 * la + 1 : (la + 1) * (la + 2) / 2;
  const int nb = sh.pure && lb > 1 ? 2 * lb + 1 : (lb + 1) * (lb + 2) / 2;
  int X = la * (la + 1) / 2 + lb, off = 0;
  for (int k = 0; k < X; ++k) off += ix.cnt[k];
  const bool diag = pr.sa[P] == pr.sb[P];  // both orders are components of the block: the one with i >= j counts
  for (int i = 0; i < na; ++i)
    for (int j = 0; j < nb; ++j) {
      if (diag && i < j) continue;
      const int row = ix.base[X] + (i * nb + j) * ix.cnt[X] + (P - off);
      const int f = sh.bfs[pr.sa[P]] + i, g = sh.bfs[pr.sb[P]] + j;
      index[(size_t)f * n + g] = row;
      index[(size_t)g * n + f] = row;
      fn[row] = max(f, g) << 16 | min(f, g);
    }
}
__global__ void k_pairm_index(QxShellsDev sh, QxPairsDev pr, int npairs, QxPairIndex ix, int* index, int* fn) {
  const int P = blockIdx.x * blockDim.x + threadIdx.x;
  if (P < npairs) pairm_index(sh, pr, P, ix, index, fn);
}

// The tables of a small context and its cleared matrices in one workgroup:
// launches are most of such a tensor's time (two functions: 57 us with
// three launches more, 27 us).
#define PM_SMALL 16384  // doubles of the matrices, ints of the tables
__global__ __launch_bounds__(512) void k_pairm_small(QxShellsDev sh, QxPairsDev pr, int npairs, QxPairIndex ix, int ld,
                                                     int* index, int* fn, double* M, int nm) {
  for (int i = threadIdx.x; i < sh.nbf * sh.nbf; i += blockDim.x) index[i] = -1;
  for (int i = threadIdx.x; i < ld; i += blockDim.x) fn[i] = -1;
  for (int i = threadIdx.x; i < nm; i += blockDim.x) M[i] = 0.0;
  __syncthreads();
  for (int P = threadIdx.x; P < npairs; P += blockDim.x) pairm_index(sh, pr, P, ix, index, fn);
}

// Class and pair position of row r.
__device__ __forceinline__ void pairm_row(const QxPairIndex& ix, int r, int& X, int& pos) {
  X = 0;
#pragma unroll
  for (int k = 1; k < 6; ++k) X = r >= ix.base[k] ? k : X;
  pos = (r - ix.base[X]) % max(ix.cnt[X], 1);
}

// Cartesian components of a shell pair to solid-harmonic ones, in place.
template <int LA, int LB>
__device__ __forceinline__ void pm_to_ao(double* m, size_t step, const double* sph) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2, MA = 2 * LA + 1, MB = 2 * LB + 1;
  double v[NA * NB];
#pragma unroll
  for (int k = 0; k < NA * NB; ++k) v[k] = m[k * step];
#pragma unroll
  for (int i = 0; i < MA; ++i) {
    double w[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      w[q] = LA == 2 ? 0.0 : v[i * NB + q];
      if (LA == 2) {
#pragma unroll
        for (int k = 0; k < NA; ++k) w[q] += sph[i * 6 + k] * v[k * NB + q];
      }
    }
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      double z = LB == 2 ? 0.0 : w[j];
      if (LB == 2) {
#pragma unroll
        for (int k = 0; k < NB; ++k) z += sph[j * 6 + k] * w[k];
      }
      m[(i * MB + j) * step] = z;
    }
  }
}
__device__ __forceinline__ void pm_to_ao(int X, double* m, size_t step, const double* sph) {
  if (X == 3) pm_to_ao<2, 0>(m, step, sph);
  else if (X == 4) pm_to_ao<2, 1>(m, step, sph);
  else pm_to_ao<2, 2>(m, step, sph);
}

// The stored half of a spherical context's M to AO components: KET, columns of
// the pairs with a d shell in every row; then rows.  One lane per (row, ket
// pair) or (bra pair, column), consecutive lanes on consecutive columns: two
// passes over the half that has d shells, bound by HBM.
template <bool KET>
__global__ __launch_bounds__(256) void k_pairm_ao(QxShellsDev sh, QxPairIndex ix, const int* fn, double* M, long long ld,
                                                  long long slice) {
  __shared__ double sph[30];
  if (threadIdx.x < 30) sph[threadIdx.x] = sh.sph[sh.sph_off[2] + threadIdx.x];
  __syncthreads();
  M += (long long)blockIdx.z * slice;
  const int lane = blockIdx.x * 256 + threadIdx.x;
  // position i of the pairs with a d shell: class and place in it
  auto pair = [&](int i, int& X, int& pos) {
    X = i < ix.cnt[3] ? 3 : i < ix.cnt[3] + ix.cnt[4] ? 4 : 5;
    pos = i - (X > 3 ? ix.cnt[3] : 0) - (X > 4 ? ix.cnt[4] : 0);
  };
  const int nd = ix.cnt[3] + ix.cnt[4] + ix.cnt[5];
  int X, pos, Y, j;
  if (KET) {
    if (lane >= nd) return;
    pair(lane, Y, j);
    for (int r = ix.base[Y] + (int)blockIdx.y; r < ix.base[6]; r += gridDim.y) {
      pairm_row(ix, r, X, pos);
      if (X == Y && pos < j) continue;  // the mirrored half
      pm_to_ao(Y, M + (long long)r * ld + ix.base[Y] + j, ix.cnt[Y], sph);
    }
  } else {
    if (lane >= ix.base[6] || fn[lane] < 0) return;
    pairm_row(ix, lane, Y, j);
    for (int i = blockIdx.y; i < nd; i += gridDim.y) {
      pair(i, X, pos);
      if (Y > X || (Y == X && j > pos)) continue;
      pm_to_ao(X, M + (long long)(ix.base[X] + pos) * ld + lane, (size_t)ix.cnt[X] * ld, sph);
    }
  }
}

// The quartet kernels store (row, column) for bra class > ket class, or bra
// position >= ket position within a class; the other elements are the
// transposed ones.  A workgroup owns the 32 x 32 tile (tr, tc) and its mirror
// image, so it reads what it needs of both before it writes either: of a tile
// between two classes, only the stored half.  Bound by HBM (half of M read and
// written).  Tiles of 64 with the class of every element worked out by each
// lane took 402 us for the 112-function tensor's 0.4 GB, this takes 105.
#define PM_TILE 32
__global__ __launch_bounds__(256) void k_pairm_sym(double* M, long long ld, long long slice, QxPairIndex ix) {
  __shared__ double a[PM_TILE][PM_TILE + 1], b[PM_TILE][PM_TILE + 1];
  __shared__ int cls[2 * PM_TILE], pos[2 * PM_TILE];  // of the tile's rows, then of its columns
  M += (long long)blockIdx.y * slice;
  const long long t = blockIdx.x;
  int tr = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(tr + 1) * (tr + 2) / 2 <= t) ++tr;
  while ((long long)tr * (tr + 1) / 2 > t) --tr;
  const int tc = (int)(t - (long long)tr * (tr + 1) / 2);
  const int r0 = tr * PM_TILE, c0 = tc * PM_TILE;
  const int lx = threadIdx.x % PM_TILE, ly = threadIdx.x / PM_TILE, step = 256 / PM_TILE;
  if (threadIdx.x < 2 * PM_TILE) pairm_row(ix, ly == 0 ? r0 + lx : c0 + lx, cls[threadIdx.x], pos[threadIdx.x]);
  __syncthreads();
  const bool whole = cls[0] > cls[2 * PM_TILE - 1];  // rows of higher classes than every column: the tile is stored
  for (int y = ly; y < PM_TILE; y += step) {
    a[y][lx] = r0 + y < ld && c0 + lx < ld ? M[(long long)(r0 + y) * ld + c0 + lx] : 0.0;
    if (!whole) b[y][lx] = c0 + y < ld && r0 + lx < ld ? M[(long long)(c0 + y) * ld + r0 + lx] : 0.0;
  }
  __syncthreads();
  auto there = [&](int r, int c) { return cls[r] > cls[c] || (cls[r] == cls[c] && pos[r] >= pos[c]); };
  for (int y = ly; y < PM_TILE; y += step) {
    if (!whole && r0 + y < ld && c0 + lx < ld && !there(y, PM_TILE + lx)) M[(long long)(r0 + y) * ld + c0 + lx] = b[lx][y];
    if (c0 + y < ld && r0 + lx < ld && tr != tc && !there(PM_TILE + y, lx))
      M[(long long)(c0 + y) * ld + r0 + lx] = a[lx][y];
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
  if (pq < 0 || rs < 0) return;
  const size_t n = nc, p = pq >> 16, q = pq & 0xffff, r = rs >> 16, u = rs & 0xffff;
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

// One workgroup per AO function pair p >= q (and slice, and panel of rows r):
// the row of (p, q) is put in LDS as the triangle r >= u (TRI) or as the
// panel's rows, and then written to out[p][q] and out[q][p].  Bound by the
// tensor's HBM writes.  Transforming to AO functions here, with a gather
// through an index table per (r, u), took 1196 us for the 112-function tensor
// (1.26 GB), with one lane per ket shell pair 822 us; this takes 330 and the
// two transforming passes 125.  HALF: M is not mirrored, an element of the other
// half is read where it is stored (small matrices: a launch less).
#define PM_HALF 512  // rows
#define PM_LDS_TRI (150 * 1024)  // a triangle takes one panel up to here (n <= 195)
#define PM_LDS_ROWS (72 * 1024)  // rows of a panel beyond: two workgroups per CU
// An output row pair goes out without a stay in the caches: nothing reads it here.
typedef double pm_dv2 __attribute__((vector_size(16)));
template <bool TRI, bool HALF>
__global__ __launch_bounds__(1024) void k_pairm_expand(int n, const double* M, long long ld, long long slice, QxPairIndex ix,
                                                      const int* index, const int* fn, int rows, double* out) {
  HIP_DYNAMIC_SHARED(double, row)
  const long long t = blockIdx.x;
  int p = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((long long)(p + 1) * (p + 2) / 2 <= t) ++p;
  while ((long long)p * (p + 1) / 2 > t) --p;
  const int q = (int)(t - (long long)p * (p + 1) / 2);
  const int r0 = TRI ? 0 : (int)blockIdx.z * rows, r1 = TRI ? n : min(n, r0 + rows);
  const int len = TRI ? n * (n + 1) / 2 : (r1 - r0) * n;
  for (int k = threadIdx.x; k < len; k += blockDim.x) row[k] = 0.0;  // pairs that the screening dropped
  __syncthreads();
  const int from = index[(size_t)p * n + q];
  if (from >= 0) {
    const double* m = M + (long long)blockIdx.y * slice + from * ld;
    int X = 0, pos = 0;
    if (HALF) pairm_row(ix, from, X, pos);
#pragma unroll 4
    for (int c = threadIdx.x; c < ld; c += blockDim.x) {
      const int f = fn[c], r = f >> 16, u = f & 0xffff;
      if (f < 0) continue;
      double v;
      if (HALF) {
        int Y, j;
        pairm_row(ix, c, Y, j);
        v = X > Y || (X == Y && pos >= j) ? m[c] : M[(long long)blockIdx.y * slice + c * ld + from];
      } else {
        v = m[c];
      }
      if (TRI) {
        row[r * (r + 1) / 2 + u] = v;
      } else {
        if (r >= r0 && r < r1) row[(r - r0) * n + u] = v;
        if (u >= r0 && u < r1) row[(u - r0) * n + r] = v;
      }
    }
  }
  __syncthreads();
  const long long nn = (long long)n * n;
  double* const o1 = out + (long long)blockIdx.y * nn * nn + ((long long)p * n + q) * nn;
  double* const o2 = out + (long long)blockIdx.y * nn * nn + ((long long)q * n + p) * nn;
  const int lane = threadIdx.x & 63;
  const bool wide = n % 2 == 0 && (reinterpret_cast<size_t>(out) & 15) == 0;
  for (int r = r0 + (int)(threadIdx.x >> 6); r < r1; r += (int)(blockDim.x >> 6)) {
    auto at = [&](int u) {
      if (TRI) return u <= r ? row[r * (r + 1) / 2 + u] : row[u * (u + 1) / 2 + r];
      return row[(r - r0) * n + u];
    };
    const long long o = (long long)r * n;
    if (wide) {
      for (int u = 2 * lane; u < n; u += 128) {
        const pm_dv2 v = {at(u), at(u + 1)};
        __builtin_nontemporal_store(v, reinterpret_cast<pm_dv2*>(o1 + o + u));
        if (p != q) __builtin_nontemporal_store(v, reinterpret_cast<pm_dv2*>(o2 + o + u));
      }
    } else {
      for (int u = lane; u < n; u += 64) {
        const double v = at(u);
        o1[o + u] = v;
        if (p != q) o2[o + u] = v;
      }
    }
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

int qxk_pairm_tables(const QxShellsDev* sh, const QxPairsDev* pr, int npairs, const QxPairIndex* ix, long long ld, int* index,
                     int* fn, double* M, long long nm, int* cleared, hipStream_t s) {
  const long long n2 = (long long)sh->nbf * sh->nbf;
  *cleared = n2 + ld <= PM_SMALL && nm <= PM_SMALL;
  if (*cleared) {
    hipLaunchKernelGGL(k_pairm_small, dim3(1), dim3(512), 0, s, *sh, *pr, npairs, *ix, (int)ld, index, fn, M, (int)nm);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(k_fill_int, dim3(std::min(nblk(n2, 256), 4096u)), dim3(256), 0, s, index, n2, -1);
  hipLaunchKernelGGL(k_fill_int, dim3(std::min(nblk(ld, 256), 4096u)), dim3(256), 0, s, fn, ld, -1);
  if (npairs > 0)
    hipLaunchKernelGGL(k_pairm_index, dim3(nblk(npairs, 64)), dim3(64), 0, s, *sh, *pr, npairs, *ix, index, fn);
  return (int)hipGetLastError();
}

int qxk_pairm_ao(const QxShellsDev* sh, const QxPairIndex* ix, const int* fn, double* M, long long ld, long long slice,
                 int nslice, hipStream_t s) {
  const int nd = ix->cnt[3] + ix->cnt[4] + ix->cnt[5];
  if (!sh->pure || nd <= 0 || nslice <= 0) return 0;
  if (nslice > 65535) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pairm_ao<true>, dim3(nblk(nd, 256), (unsigned)std::min(ix->base[6], 65535), (unsigned)nslice),
                     dim3(256), 0, s, *sh, *ix, fn, M, ld, slice);
  hipLaunchKernelGGL(k_pairm_ao<false>, dim3(nblk(ix->base[6], 256), (unsigned)std::min(nd, 65535), (unsigned)nslice),
                     dim3(256), 0, s, *sh, *ix, fn, M, ld, slice);
  return (int)hipGetLastError();
}

// Whether the expansion reads the stored half (M is then not mirrored).
static bool pairm_half(int n, long long ld) {
  return ld <= PM_HALF && (size_t)n * (n + 1) / 2 * sizeof(double) <= PM_LDS_TRI;
}

int qxk_pairm_sym(int n, double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix, hipStream_t s) {
  const long long T = (ld + PM_TILE - 1) / PM_TILE, tiles = T * (T + 1) / 2;
  if (tiles <= 0 || nslice <= 0 || pairm_half(n, ld)) return 0;
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

int qxk_pairm_expand(int n, const double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix,
                     const int* index, const int* fn, double* out, hipStream_t s) {
  if (nslice <= 0) return 0;
  const size_t tri = (size_t)n * (n + 1) / 2 * sizeof(double);
  const bool one = tri <= PM_LDS_TRI;
  const int rows = one ? n : (int)std::max<size_t>(1, PM_LDS_ROWS / ((size_t)n * sizeof(double)));
  const size_t bytes = one ? tri : (size_t)rows * n * sizeof(double);
  const dim3 grid((unsigned)((long long)n * (n + 1) / 2), (unsigned)nslice, (unsigned)((n + rows - 1) / rows));
  if (nslice > 65535 || bytes > PM_LDS_TRI) return (int)hipErrorInvalidValue;
  // 256 / 512 / 1024 threads in us: 28 functions 7 / 6 / 7 (three slices 8 / 9 / 12), 56 functions 19 / 17.5 / 19,
  // 84 functions 103 / 96 / 94, 92 functions 137 / 132 / 126, 112 functions 441 / 359 / 310
  const dim3 block(n < 64 ? 512 : 1024);
  if (pairm_half(n, ld)) hipLaunchKernelGGL((k_pairm_expand<true, true>), grid, block, bytes, s, n, M, ld, slice, *ix, index, fn, rows, out);
  else if (one) hipLaunchKernelGGL((k_pairm_expand<true, false>), grid, block, bytes, s, n, M, ld, slice, *ix, index, fn, rows, out);
  else hipLaunchKernelGGL((k_pairm_expand<false, false>), grid, block, bytes, s, n, M, ld, slice, *ix, index, fn, rows, out);
  return (int)hipGetLastError();
}

int qxk_oei_deriv(const QxShellsDev* sh, double* dS, double* dT, double* dV, hipStream_t s) {
  const unsigned rows = (unsigned)std::min(sh->natom + 1, 65535);
  hipLaunchKernelGGL(k_oei_deriv, dim3(nblk((long long)sh->nshell * sh->nshell, 64), rows), dim3(64), 0, s, *sh, dS, dT,
                     dV);
  return (int)hipGetLastError();
}

}  // extern "C"
