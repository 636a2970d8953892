// Adjoint gradient: each derivative integral is contracted with the density
// pair product when formed.  A workgroup owns one bra pair and a run of its
// kets (the K kernels' decomposition), so the bra centres' terms stay in
// registers for the whole run; the ket centres' terms go to LDS accumulators
// over the block's atom window and reach the global gradient once per block.
#pragma once
#include "qx_jk.h"

// Gradient accumulators of a workgroup: a window of atoms in LDS, or its copy
// of the global gradient.
struct QxGradTarget {
  double* sg;      // LDS window, or null
  double* g;       // the block's copy of the global gradient
  int lo, w;       // window: 3 * first atom, doubles
  __device__ __forceinline__ void add(int slot, double v) const {
    if (sg) atomicAdd(&sg[slot - lo], v);
    else qx_atomic_add(&g[slot], v);
  }
};
__device__ __forceinline__ QxGradTarget qx_grad_begin(const QxArgs& A_, const QxKList& kl, int P1, double* lds) {
  QxGradTarget t;
  const int nc = A_.e.grad_copies > 1 ? A_.e.grad_copies : 1;
  t.g = A_.e.grad + (size_t)((blockIdx.x + blockIdx.y * 7 + blockIdx.z * 13) % nc) * (size_t)(3 * A_.e.natom);
  const int cap = A_.e.grad_win > 0 && A_.e.grad_win < QX_GRAD_LDS ? A_.e.grad_win : QX_GRAD_LDS;
  t.lo = 0;
  t.w = 3 * A_.e.natom;
  if (kl.frag_atoms && t.w > cap) {  // every centre of the block lies in its bra's fragment
    const int f = A_.e.pair_frag[P1];
    t.lo = 3 * kl.frag_atoms[2 * f];
    t.w = 3 * kl.frag_atoms[2 * f + 1];
  }
  t.sg = t.w <= cap ? lds : nullptr;
  if (t.sg)
    for (int i = threadIdx.x; i < t.w; i += blockDim.x) lds[i] = 0.0;
  __syncthreads();
  return t;
}
__device__ __forceinline__ void qx_grad_end(const QxGradTarget& t) {
  __syncthreads();
  if (!t.sg) return;
  for (int i = threadIdx.x; i < t.w; i += blockDim.x)
    if (t.sg[i] != 0.0) qx_atomic_add(&t.g[t.lo + i], t.sg[i]);
}
// The bra centres' sums of every lane (all kets of the block), once per block.
__device__ __forceinline__ void qx_grad_bra(const QxArgs& A_, const QxGradTarget& t, int P1, const double (&g)[6]) {
  const int at[2] = {A_.pr.atom_a[P1], A_.pr.atom_b[P1]};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    if (A_.e.grad_wred) {  // launch-uniform
      const double v = qx_wave_sum(g[k]);
      if (__lane_id() == 0) t.add(3 * at[k / 3] + k % 3, v);
    } else {
      t.add(3 * at[k / 3] + k % 3, g[k]);
    }
  }
}


// Light classes: one lane (or kl.sub lanes, which share the primitives) per
// contracted quartet; part(P1, P2, u1, u2, g) adds one primitive quartet's
// d/dA, d/dB, d/dC sums.
#define QX_GRAD_NCOMB 9
template <class Part>
__device__ __forceinline__ void qx_grad_block(const QxArgs& A_, const QxKList& kl, const QxKBlock& b, double* sg, Part part) {
  const QxGradTarget tgt = qx_grad_begin(A_, kl, b.P1, sg);
  const int u1 = A_.pr.pp_first[b.P1], n1 = A_.pr.pp_n[b.P1];
  double gb[6] = {};
  for (int t = (int)threadIdx.x; t < (b.j1 - b.j0) * kl.sub; t += (int)blockDim.x) {
    const int P2 = b.kst + b.j0 + t / kl.sub;
    if (qx_single_atom(A_, b.P1, P2)) continue;
    const int u2 = A_.pr.pp_first[P2], n2 = A_.pr.pp_n[P2];
    double g[QX_GRAD_NCOMB] = {};
    for (int k = t % kl.sub; k < n1 * n2; k += kl.sub) part(b.P1, P2, u1 + k / n2, u2 + k % n2, g);
    const double w = 8.0 * qx_degeneracy(A_, b.P1, P2);
    const int atc = 3 * A_.pr.atom_a[P2], atd = 3 * A_.pr.atom_b[P2];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double a = w * g[x], bb = w * g[3 + x], c = w * g[6 + x];
      gb[x] += a;
      gb[3 + x] += bb;
      tgt.add(atc + x, c);
      tgt.add(atd + x, -(a + bb + c));
    }
  }
  qx_grad_bra(A_, tgt, b.P1, gb);
  qx_grad_end(tgt);
}

// Launcher of a generated kernel qx_kg_NAME.
#define QX_DEFINE_GRAD_LAUNCHER(NAME, WITH32)                                                     \
  extern "C" int qx_launchg_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    const int bs = qx_launch_block(L);                                                            \
    if (bs % 64 || bs > QX_BLOCK_MAX) return (int)hipErrorInvalidValue;                           \
    const QxKList& kl = *L->kl;                                                                   \
    const dim3 grid((unsigned)kl.nbra, (unsigned)((kl.maxket + kl.chunk - 1) / kl.chunk));        \
    if (L->fp32) {                                                                                \
      if constexpr (WITH32) hipLaunchKernelGGL(qx_kg_##NAME<float>, grid, dim3(bs), 0, L->stream, *a, kl); \
      else return -1;                                                                             \
    } else {                                                                                      \
      hipLaunchKernelGGL(qx_kg_##NAME<double>, grid, dim3(bs), 0, L->stream, *a, kl);             \
    }                                                                                             \
    return (int)hipGetLastError();                                                                \
  }

// Launcher of the generated kernels of a class's directional derivative.
#define QX_DEFINE_GRADV_LAUNCHER(NAME, ...)                                                       \
  extern "C" int qx_launchh_##NAME(const QxArgs* a, const QxLaunch* L) {                          \
    if (!L->kl || L->kl->nquart <= 0 || L->kl->maxket <= 0) return 0;                             \
    const int bs = qx_launch_block(L);                                                            \
    if (bs % 64 || bs > QX_BLOCK_MAX) return (int)hipErrorInvalidValue;                           \
    if (!a->e.tv) return -1;                                                                      \
    const QxKList& kl = *L->kl;                                                                   \
    const dim3 grid((unsigned)kl.nbra, (unsigned)((kl.maxket + kl.chunk - 1) / kl.chunk));        \
    for (auto kernel : {__VA_ARGS__}) hipLaunchKernelGGL(kernel, grid, dim3(bs), 0, L->stream, *a, kl); \
    return (int)hipGetLastError();                                                                \
  }

// Every gradient kernel of a context without d shells in one launch (as
// qx_small of the J/K pass): QX_SMALL_GRADS of them, each a class's list.
struct QxSmallGrad {
  QxKList k[6];  // per class: 0000, 1000, 1010, 1100, 1110, 1111
  int end[16];   // workgroups of the kernels up to each one
};
