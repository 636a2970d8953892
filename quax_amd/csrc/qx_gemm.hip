// FP64 MFMA GEMM for the AO -> MO integral transformation (reference:
// quax/methods/energy_utils.py:46-73; callers mp2.py:29, ccsd.py:32).
//
// One transformation step contracts the last index of a row-major tensor X
// (R rows of n) with a coefficient matrix C (n x m, row-major) and puts the
// new index first:  Y[M, r] = sum_s C[s, M] X[r, s]  -- the reference's
// jnp.tensordot(C, X, axes=[(0,), (3,)]).  As a GEMM, Y (m x R) = C^T X^T:
// both operands are read "transposed", which the kernel does directly from
// LDS tiles (no transposed copies).
//
// Kernel: all of up to 128 rows of Y (MT tiles of 16, no padding beyond the
// last one) x 128 columns per 256-thread workgroup, so X is read once: wave w
// owns 32 columns and every row (MT x 2 tiles of v_mfma_f64_16x16x4f64).  K
// goes in steps of 16 through two LDS buffers: the next step is loaded into
// registers before the current one is multiplied and stored to the other
// buffer after it, one barrier per step.  MFMA operand layout (16x16x4, FP64,
// checked on gfx950 with a one-wavefront probe): lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16]; accumulator element r of lane l is
// D[4 r + l / 16][l % 16] (rows interleaved across the four 16-lane groups).
// Bound by the FP64 matrix rate (2 M flops per 8 bytes of X; 68-72 TFLOP/s
// reached by a large product on this part) and HBM together: at 112 functions
// one quarter is 0.45 ms of products and 0.55 ms of reading and writing, which
// overlap to 0.81-0.94 ms (9.05 -> 3.2 ms for all four against 64 x 64 tiles
// staged step by step).  Keeping C in LDS under persistent workgroups,
// contiguous output orientations without barriers, deeper prefetch and slices
// that stay in the last-level cache gave 3.26-3.6 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "quax_amd.h"

namespace {

typedef double qx_dv4 __attribute__((ext_vector_type(4)));

constexpr int GM_BK = 16, GM_THREADS = 256;
constexpr int GM_BS = GM_BK + 2;  // B row stride: 16 rows x 4 k hit distinct LDS banks

// out[i * ldo + j] = sum_k A[k * lda + i] B[j * ldb + k], i < M, j < N, k < K,
// for the rows i0 = blockIdx.y * 16 MT onwards and NT * 64 columns.
template <int MT, int NT>
__global__ __launch_bounds__(GM_THREADS) void qx_dgemm_tt_kernel(int M, long long N, int K, const double* __restrict__ A,
                                                                  long long lda, const double* __restrict__ B,
                                                                  long long ldb, double* __restrict__ out,
                                                                  long long ldo) {
  constexpr int BM = 16 * MT, BN = 64 * NT;
  constexpr int AS = BM + (MT % 2 ? 0 : 16);  // odd multiple of 16: the two k of a half wave hit distinct banks
  constexpr int NA = (GM_BK * BM + GM_THREADS - 1) / GM_THREADS, NB = GM_BK * BN / GM_THREADS;
  __shared__ double As[2][GM_BK * AS];
  __shared__ double Bs[2][BN * GM_BS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = (int)blockIdx.y * BM;
  const long long j0 = (long long)blockIdx.x * BN;
  qx_dv4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = qx_dv4{0.0, 0.0, 0.0, 0.0};
  double ra[NA], rb[NB];
  auto load = [&](int k0) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int idx = tid + r * GM_THREADS, k = idx / BM, i = idx - k * BM;
      ra[r] = k < GM_BK && i0 + i < M && k0 + k < K ? A[(long long)(k0 + k) * lda + i0 + i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int idx = tid + r * GM_THREADS, j = idx / GM_BK, k = idx % GM_BK;
      rb[r] = j0 + j < N && k0 + k < K ? B[(j0 + j) * ldb + k0 + k] : 0.0;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int idx = tid + r * GM_THREADS, k = idx / BM, i = idx - k * BM;
      if (k < GM_BK) As[buf][k * AS + i] = ra[r];
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int idx = tid + r * GM_THREADS, j = idx / GM_BK, k = idx % GM_BK;
      Bs[buf][j * GM_BS + k] = rb[r];
    }
  };
  load(0);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += GM_BK, buf ^= 1) {
    const bool more = k0 + GM_BK < K;
    if (more) load(k0 + GM_BK);
    const int kc = min(GM_BK, K - k0);
    for (int kk = 0; kk < kc; kk += 4) {  // block-uniform
      const int ka = kk + (lane >> 4);
      double b[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) b[t] = Bs[buf][(wave * 16 * NT + t * 16 + (lane & 15)) * GM_BS + ka];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const double a = As[buf][ka * AS + t * 16 + (lane & 15)];
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[u], acc[t][u], 0, 0, 0);
      }
    }
    if (more) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int ta = 0; ta < MT; ++ta)
#pragma unroll
    for (int tb = 0; tb < NT; ++tb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long long gi = i0 + ta * 16 + 4 * r + (lane >> 4);
        const long long gj = j0 + wave * 16 * NT + tb * 16 + (lane & 15);
        if (gi < M && gj < N) out[gi * ldo + gj] = acc[ta][tb][r];
      }
}

template <int MT>
void gemm_launch(dim3 rows, int M, long long N, int K, const double* A, const double* B, double* out, hipStream_t s) {
  // 128 columns per workgroup once that still gives every CU work, else 64
  if (N >= 128 * 512) {
    hipLaunchKernelGGL((qx_dgemm_tt_kernel<MT, 2>), dim3((unsigned)((N + 127) / 128), rows.y), dim3(GM_THREADS), 0, s, M, N,
                       K, A, (long long)M, B, (long long)K, out, N);
  } else {
    hipLaunchKernelGGL((qx_dgemm_tt_kernel<MT, 1>), dim3((unsigned)((N + 63) / 64), rows.y), dim3(GM_THREADS), 0, s, M, N, K,
                       A, (long long)M, B, (long long)K, out, N);
  }
}

thread_local std::string g_gemm_error;

int gemm_tt(int M, long long N, int K, const double* A, const double* B, double* out, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0) return QX_OK;
  const int tiles = (M + 15) / 16, gy = (tiles + 7) / 8, mt = (tiles + gy - 1) / gy;  // equal shares of at most 8 tiles
  if (gy > 65535 || (N + 63) / 64 > 0x7fffffffLL) {
    g_gemm_error = "tei transformation: tensor too large for one launch";
    return QX_EINVAL;
  }
  const dim3 rows(1, (unsigned)gy);
  switch (mt) {
    case 1: gemm_launch<1>(rows, M, N, K, A, B, out, s); break;
    case 2: gemm_launch<2>(rows, M, N, K, A, B, out, s); break;
    case 3: gemm_launch<3>(rows, M, N, K, A, B, out, s); break;
    case 4: gemm_launch<4>(rows, M, N, K, A, B, out, s); break;
    case 5: gemm_launch<5>(rows, M, N, K, A, B, out, s); break;
    case 6: gemm_launch<6>(rows, M, N, K, A, B, out, s); break;
    case 7: gemm_launch<7>(rows, M, N, K, A, B, out, s); break;
    default: gemm_launch<8>(rows, M, N, K, A, B, out, s); break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    g_gemm_error = std::string("tei transformation: ") + hipGetErrorString(e);
    return QX_EHIP;
  }
  return QX_OK;
}

}  // namespace

extern "C" {

long long qx_tei_transform_work(const int* n, const int* m) {
  if (!n || !m) return -1;
  for (int k = 0; k < 4; ++k)
    if (n[k] <= 0 || m[k] <= 0) return -1;
  const long long t1 = (long long)m[3] * n[0] * n[1] * n[2];
  const long long t2 = (long long)m[2] * m[3] * n[0] * n[1];
  const long long t3 = (long long)m[1] * m[2] * m[3] * n[0];
  return std::max(t1, t3) + t2;
}

int qx_partial_tei_transformation(const double* G, const int* n, const double* Ci, const double* Cj,
                                  const double* Ck, const double* Cl, const int* m, double* out, double* work,
                                  void* stream) {
  if (!G || !n || !m || !Ci || !Cj || !Ck || !Cl || !out || !work) {
    g_gemm_error = "tei transformation: null argument";
    return QX_EINVAL;
  }
  const long long wsize = qx_tei_transform_work(n, m);
  if (wsize < 0) {
    g_gemm_error = "tei transformation: dimensions must be positive";
    return QX_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  double* w1 = work;                                                   // T1, then T3
  double* w2 = work + std::max((long long)m[3] * n[0] * n[1] * n[2],  // T2
                               (long long)m[1] * m[2] * m[3] * n[0]);
  // T1[L, p, q, r] = sum_s Cl[s, L] G[p, q, r, s]
  int rc = gemm_tt(m[3], (long long)n[0] * n[1] * n[2], n[3], Cl, G, w1, s);
  // T2[K, L, p, q] = sum_r Ck[r, K] T1[L, p, q, r]
  if (rc == QX_OK) rc = gemm_tt(m[2], (long long)m[3] * n[0] * n[1], n[2], Ck, w1, w2, s);
  // T3[J, K, L, p] = sum_q Cj[q, J] T2[K, L, p, q]
  if (rc == QX_OK) rc = gemm_tt(m[1], (long long)m[2] * m[3] * n[0], n[1], Cj, w2, w1, s);
  // out[I, J, K, L] = sum_p Ci[p, I] T3[J, K, L, p]
  if (rc == QX_OK) rc = gemm_tt(m[0], (long long)m[1] * m[2] * m[3], n[0], Ci, w1, out, s);
  return rc;
}

const char* qx_gemm_last_error(void) { return g_gemm_error.c_str(); }

}  // extern "C"
