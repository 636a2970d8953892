// Set-up and finish of a J/K pass: Hermite densities of every primitive pair,
// J from the Hermite potential, and the Rys tables.
#include <hip/hip_runtime.h>

#include "qx_rys.h"
#include "qx_runtime.h"

namespace {

const double kRys[QX_RYS_DOUBLES] = {
#include "qx_rys.inc"
};

// One thread per pseudo pair (Hermite density); every thread also clears its
// share of the pass's accumulators, so a pass needs no fill launches.
template <typename R>
__global__ __launch_bounds__(64) void k_jk_begin(QxArgs a, QxJList jl, double* H, double* Hd, long long nherm, double* J,
                                                 double* K, long long n2) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u < jl.uoff[6]) {
    int X = 0;
#pragma unroll
    for (int k = 1; k < 6; ++k) X = u >= jl.uoff[k] ? k : X;
    switch (X) {
      case 0: qx_hermite_density<0, 0, R>(a, jl, 0, u, H, Hd); break;
      case 1: qx_hermite_density<1, 0, R>(a, jl, 1, u, H, Hd); break;
      case 2: qx_hermite_density<1, 1, R>(a, jl, 2, u, H, Hd); break;
      case 3: qx_hermite_density<2, 0, R>(a, jl, 3, u, H, Hd); break;
      case 4: qx_hermite_density<2, 1, R>(a, jl, 4, u, H, Hd); break;
      default: qx_hermite_density<2, 2, R>(a, jl, 5, u, H, Hd); break;
    }
  }
  const long long step = (long long)gridDim.x * blockDim.x;
  for (long long k = u; k < nherm; k += step) {
    jl.P[k] = 0.0;
    if (a.e.tv) jl.Pd[k] = 0.0;
  }
  for (long long k = u; k < n2; k += step) {
    J[k] = 0.0;
    K[k] = 0.0;
  }
}

// One thread per contracted pair: its J block.
template <typename R>
__global__ __launch_bounds__(64) void k_j_finish(QxArgs a, QxJList jl, double* J) {
  const int P = blockIdx.x * blockDim.x + threadIdx.x;
  if (P >= jl.npairs) return;
  const int u = a.pr.pp_first[P];
  int X = 0;
#pragma unroll
  for (int k = 1; k < 6; ++k) X = u >= jl.uoff[k] ? k : X;
  switch (X) {
    case 0: qx_hermite_potential<0, 0, R>(a, jl, 0, P, J); break;
    case 1: qx_hermite_potential<1, 0, R>(a, jl, 1, P, J); break;
    case 2: qx_hermite_potential<1, 1, R>(a, jl, 2, P, J); break;
    case 3: qx_hermite_potential<2, 0, R>(a, jl, 3, P, J); break;
    case 4: qx_hermite_potential<2, 1, R>(a, jl, 4, P, J); break;
    default: qx_hermite_potential<2, 2, R>(a, jl, 5, P, J); break;
  }
}

// AO J and K from the Cartesian J and the unsymmetrised K' (grid row 0 / 1):
// T J T^T and T (K' + K'^T) / 2 T^T, T = 1 for a Cartesian basis.
__global__ void k_jk_finish(QxShellsDev sh, const double* Jc, const double* Kp, double* J, double* K) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = sh.nbf, nc = sh.ncart;
  if (t >= (long long)nb * nb) return;
  const int i = (int)(t / nb), j = (int)(t % nb);
  const bool k = blockIdx.y == 1;
  const double* X = k ? Kp : Jc;
  auto at = [&](int p, int q) {
    const double v = X[(size_t)p * nc + q];
    return k ? 0.5 * (v + X[(size_t)q * nc + p]) : v;
  };
  double acc = 0.0;
  if (!sh.pure) {
    acc = at(i, j);
  } else {
    const int si = sh.ao_shell[i], sj = sh.ao_shell[j];
    const int li = sh.l[si], lj = sh.l[sj];
    const int ni = (li + 1) * (li + 2) / 2, nj = (lj + 1) * (lj + 2) / 2;
    const double* ti = sh.sph + sh.sph_off[li] + (i - sh.bfs[si]) * ni;
    const double* tj = sh.sph + sh.sph_off[lj] + (j - sh.bfs[sj]) * nj;
    for (int p = 0; p < ni; ++p) {
      if (ti[p] == 0.0) continue;
      for (int q = 0; q < nj; ++q)
        if (tj[q] != 0.0) acc += ti[p] * tj[q] * at(sh.bfc[si] + p, sh.bfc[sj] + q);
    }
  }
  (k ? K : J)[t] = acc;
}

}  // namespace

extern "C" {

const double* qxk_rys_host(void) { return kRys; }

int qxk_jk_begin(const QxArgs* a, const QxJList* jl, long long nherm, double* J, double* K, long long n2,
                 hipStream_t s) {
  const dim3 nb((unsigned)std::max<long long>((jl->uoff[6] + 63) / 64, 1));
  double *H = const_cast<double*>(jl->H), *Hd = const_cast<double*>(jl->Hd);
  if (a->e.tv) hipLaunchKernelGGL(k_jk_begin<qx_dual>, nb, dim3(64), 0, s, *a, *jl, H, Hd, nherm, J, K, n2);
  else hipLaunchKernelGGL(k_jk_begin<double>, nb, dim3(64), 0, s, *a, *jl, H, Hd, nherm, J, K, n2);
  return (int)hipGetLastError();
}

int qxk_j_finish(const QxArgs* a, const QxJList* jl, double* J, hipStream_t s) {
  if (jl->npairs <= 0) return 0;
  const dim3 nb((unsigned)((jl->npairs + 63) / 64));
  if (a->e.tv) hipLaunchKernelGGL(k_j_finish<qx_dual>, nb, dim3(64), 0, s, *a, *jl, J);
  else hipLaunchKernelGGL(k_j_finish<double>, nb, dim3(64), 0, s, *a, *jl, J);
  return (int)hipGetLastError();
}

int qxk_jk_finish(const QxShellsDev* sh, const double* Jc, const double* Kp, double* J, double* K, hipStream_t s) {
  const long long n2 = (long long)sh->nbf * sh->nbf;
  hipLaunchKernelGGL(k_jk_finish, dim3((unsigned)((n2 + 255) / 256), 2), dim3(256), 0, s, *sh, Jc, Kp, J, K);
  return (int)hipGetLastError();
}

}  // extern "C"
