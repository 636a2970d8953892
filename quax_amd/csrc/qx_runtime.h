// Host-side context of the ERI library and the helper-kernel entry points
// shared between qx_runtime.hip and qx_kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "qx_device.h"
#include "qx_jk.h"
#include "qx_pairm.h"

#define QX_LMAX_SUPPORTED 2

// Per-shell and per-function tables for the one-electron kernels and the
// spherical transforms.
struct QxShellsDev {
  int nshell, natom, ncart, nbf;
  const int* l; const int* atom; const int* nprim; const int* poff;
  const int* bfc;                         // first Cartesian function of each shell
  const int* bfs;                         // first AO (spherical when pure) function
  const double* exps; const double* coefs;
  const double* xyz;                      // 3*natom
  const double* Z;                        // natom
  const int* f_shell;                     // Cartesian function -> shell
  const int* f_comp;                      // Cartesian function -> packed (lx,ly,lz)
  const int* ao_shell;                    // AO function -> shell
  const double* sph;                      // per-l transform blocks, offsets below
  int sph_off[QX_LMAX_SUPPORTED + 2];
  int pure;
};

struct QxWorkHost {
  int cls;                 // canonical class index into the kernel table
  int bra_class, ket_class;
  QxWorkDev w;             // device view (prefix/kstart point into ctx buffers)
  long long prefix_off;    // offset of this list's prefix in ctx->d_prefix
  // the same list over contracted pairs: running counts per bra pair in
  // ctx->d_cprefix and (fragmented contexts) first kets in ctx->d_ckstart
  long long cprefix_off;
  long long ncq;           // contracted quartets
  int prims;               // primitive quartets of one (mean, rounded up)
  int maxket;              // most kets of one bra pair
};

// Row/column index of the pair matrix (qx_pairm.h): pair class X holds
// rows base[X] + component * cnt[X] + (pair position in X).
struct QxPairIndex {
  int base[7];
  int cnt[6];
};

#define QX_NUM_CLASSES_MAX 21  // canonical classes with l <= 2

struct qx_ctx {
  int device = 0;
  int natom = 0;
  std::vector<double> xyz, Z;
  int nshell = 0;
  std::vector<int> l, atom, nprim, poff, bfc, bfs;
  std::vector<double> exps, coefs;
  int pure = 0, nbf = 0, ncart = 0;
  double tol = 1e-12;
  bool k1 = true;          // every shell has one primitive
  // fragment of each atom: shell pairs and quartets never mix fragments, so
  // one context (and one launch per class) serves a batch of molecules
  std::vector<int> frag;
  bool fragmented = false;
  std::string err;

  // device memory owned by the context
  std::vector<void*> allocs;
  double* d_boys = nullptr;
  QxShellsDev shells{};
  int* d_shell_by_l = nullptr;           // shells grouped by l; group l is [l_off[l], l_off[l + 1])
  int l_off[QX_LMAX_SUPPORTED + 2] = {};
  // screened pairs + pseudo pairs (sorted)
  QxPairsDev pr{};
  QxPrimPairsDev pp{};
  int npairs = 0, npseudo = 0;
  std::vector<double> Q;                 // Schwarz value per shell pair (ns*ns)
  std::vector<int> ref_pairs;            // reference-order screened pair list
  // host copies of the sorted screened pairs
  std::vector<int> h_pair_sa, h_pair_sb, h_pair_class, h_pp_first, h_pp_n;
  std::vector<double> h_pair_Q;
  std::vector<int> h_pair_frag;
  std::vector<int> class_pair_off, class_pair_cnt;   // per pair class, in sorted pairs
  std::vector<int> class_prims;                      // per pair class: most primitives of a pair
  // quartet lists (one per canonical class)
  std::vector<QxWorkHost> work;
  long long* d_prefix = nullptr;
  int* d_kstart = nullptr;               // per bra pseudo pair, fragmented contexts only
  long long* d_cprefix = nullptr;        // running contracted quartet counts per bra pair of every list
  int* d_ckstart = nullptr;              // per bra pair (d_cprefix's offsets), fragmented contexts only
  // J kernels: admissible pseudo kets of every pair in every class, the
  // Hermite densities and potentials (value and derivative parts: 4 arrays of
  // nherm doubles) and their layout; Rys tables of the K kernels
  QxRange* d_range = nullptr;
  QxJList jlist{};
  double* d_herm = nullptr;
  double* d_herm_own = nullptr;          // value parts (H, P) of qx_jk_build_noalloc
  long long nherm = 0;
  double* d_rys = nullptr;
  // pair-matrix workspace of the tensor entry points, kept up to
  // QX_PAIRM_KEEP bytes (and pairm_limit); passes that use it are ordered like
  // those on ws
  double* pairm = nullptr;
  size_t pairm_bytes = 0;
  size_t pairm_limit = 0;                // most bytes of pair matrices per pass (0: what the device has)
  // host copies of the list arrays (quartet -> pair maps for callers that
  // read the stored integrals) and of the pseudo pair -> pair map
  std::vector<long long> h_prefix;
  std::vector<long long> h_cprefix;
  std::vector<int> h_kstart;             // per bra pseudo pair of every list
  std::vector<long long> h_kstart_off;   // per list: offset into h_kstart
  std::vector<int> h_ppair;
  long long nquart_total = 0;            // canonical contracted quartets
  long long npq_total = 0;               // pseudo-pair quartets
  long long store_total = 0;
  std::vector<long long> nq_class, ndq_class;   // contracted quartets per class (all / not single-atom)

  // optional per-kernel timing with HIP events on the launch stream
  bool profiling = false;
  struct ProfEvent {
    int slot;
    hipEvent_t start, stop;
  };
  std::vector<ProfEvent> prof_pending;
  std::vector<hipEvent_t> event_pool;
  std::vector<double> prof_ms;
  std::vector<long long> prof_launches, prof_pq;

  // independent class kernels fan out over this many streams (the caller's
  // stream plus side streams created on first use, default priority)
  int nstreams = 4;
  std::vector<hipStream_t> side;
  std::vector<hipEvent_t> fork_ev;     // [0] fork, [1..] joins

  // persistent n_cart^2 work matrices of the J/K and gradient passes (J', K',
  // Cartesian D, symmetrised J and K); ws_ev orders a pass after the previous
  // pass that used them, whatever stream each ran on
  double* ws = nullptr;
  // QX_GRAD_COPIES copies of the 3N gradient accumulators that the blocks of
  // an adjoint-gradient pass spread their flushes over (allocated on first use)
  double* gcopies = nullptr;
  // device address of the file-scope scratch array on this context's device
  // (qx_jk_build_noalloc)
  double* scratch = nullptr;
  hipEvent_t ws_ev = nullptr;
  bool ws_used = false;
  // set while a caller captures a J/K pass into a HIP graph: the pass then
  // records and waits on no event outside the capture (the graph's own
  // stream order sequences its passes)
  bool capturing = false;

  // threads per block of the streaming kernels, per pass (0 J/K, 1 adjoint
  // gradient) and class (the tuned quartet tiles)
  int tile[2][QX_NUM_CLASSES_MAX] = {};
  // per class: the adjoint-gradient kernels sum wave-uniform centres across
  // the wavefront before their LDS accumulators
  unsigned char gwred[QX_NUM_CLASSES_MAX] = {};
  // per class: copies of the gradient accumulators its blocks spread their
  // flushes over (1..QX_GRAD_COPIES)
  int gcopy[QX_NUM_CLASSES_MAX] = {};
  // per class: the J/K kernels stage K' rows in LDS (when the kernel and
  // the context allow it at all)
  unsigned char jkrows[QX_NUM_CLASSES_MAX] = {};
  // widest atom window of the adjoint kernels' LDS gradient accumulators,
  // in doubles (0: QX_GRAD_LDS)
  int grad_win = 0;
  int* d_pair_frag = nullptr;            // fragment of each sorted pair (fragmented contexts)
  // fragmented contexts: first Cartesian function of each fragment id's range
  // and the widest range (the width of the J/K kernels' LDS K' rows)
  int* d_frag_col0 = nullptr;
  int* d_frag_atoms = nullptr;           // lowest atom and window width of each fragment id
  int kcols = 0;
  // mixed precision: per class and pass (0 J/K, 1 gradient) whether quartets
  // below the threshold run in FP32 (classes whose FP32 kernels are faster)
  unsigned char fp32_ok[2][QX_NUM_CLASSES_MAX] = {};
  // the quartet lists with each bra row's FP64 ket count at one Schwarz-bound
  // threshold (kets are sorted by descending bound, so the FP64 kets of a row
  // are its first nk64 kets)
  struct Split {
    double thr = -1.0;
    std::vector<long long> pq64, pq32;   // per list: pseudo-pair quartets above / below thr
    std::vector<long long> cq64, cq32;   // per list: contracted quartets above / below thr
    int* d_ck64 = nullptr;               // FP64 kets per contracted bra pair (ctx->d_cprefix's offsets)
    int* d_range64 = nullptr;            // FP64 part of each J range (ctx->d_range's layout)
  } split;
};

// profile slots: array-form ERI kernel of class c -> QX_SLOT_ERI(c, fp32);
// derivative part / group k of class c -> QX_SLOT_DERIV(c, k, fp32); J/K
// part k of class c -> QX_SLOT_JK(c, k, fp32)
#define QX_SLOT_ERI(c, f32) ((f32) * QX_NUM_CLASSES_MAX + (c))
#define QX_SLOT_DERIV(c, k, f32) (2 * QX_NUM_CLASSES_MAX + ((f32) * QX_NUM_CLASSES_MAX + (c)) * QX_DPARTS_CAP + (k))
#define QX_SLOT_JK0 (2 * QX_NUM_CLASSES_MAX * (1 + QX_DPARTS_CAP))
#define QX_SLOT_JK(c, k, f32) (QX_SLOT_JK0 + ((f32) * QX_NUM_CLASSES_MAX + (c)) * QX_JKPARTS_CAP + (k))
#define QX_PROFILE_SLOTS (QX_SLOT_JK0 + 2 * QX_NUM_CLASSES_MAX * QX_JKPARTS_CAP)

// J/K pass set-up and finish (qx_jk.hip)
extern "C" {
const double* qxk_rys_host(void);
int qxk_jk_begin(const QxArgs* a, const QxJList* jl, long long nherm, double* J, double* K, long long n2,
                 hipStream_t s);
int qxk_j_finish(const QxArgs* a, const QxJList* jl, double* J, hipStream_t s);
int qxk_jk_finish(const QxShellsDev* sh, const double* Jc, const double* Kp, double* J, double* K, hipStream_t s);
}

// helper kernels (qx_kernels.hip)
extern "C" {
int qxk_fill(double* p, long long n, double v, hipStream_t s);
int qxk_add_copies(const double* copies, int ncopy, int n, double* out, hipStream_t s);  // out += sum of copies
int qxk_cart_to_ao_mat(const QxShellsDev* sh, const double* in, double* out, hipStream_t s);   // T X T^T
int qxk_ao_to_cart_mat(const QxShellsDev* sh, const double* in, double* out, hipStream_t s);   // T^T X T
// the same for up to three matrices in one launch; the Cartesian ones lie `stride` doubles apart
int qxk_cart_to_ao_mats(const QxShellsDev* sh, const double* in, size_t stride, double* const* out, int count,
                        hipStream_t s);
int qxk_ao_to_cart_mats(const QxShellsDev* sh, const double* const* in, double* out, size_t stride, int count,
                        hipStream_t s);
// Pair matrix M (nslice matrices of ld x ld, `slice` doubles apart) -> tensor.
// index: AO function pair -> row (nbf^2 ints, -1 = screened out), fn: row ->
// higher << 16 | lower function, -1 for none (qxk_pairm_tables fills them, and
// clears the nm doubles at M where the context is small: cleared).
int qxk_pairm_tables(const QxShellsDev* sh, const QxPairsDev* pr, int npairs, const QxPairIndex* ix, long long ld, int* index,
                     int* fn, double* M, long long nm, int* cleared, hipStream_t s);
// every permutation of the elements of a panel of rows into a zeroed
// Cartesian tensor: panel row k * cnt + i is component k of the class's pair
// i0 + i (class X, ncomp components)
int qxk_pairm_scatter(int ncart, const double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix,
                      const int* fn, int X, int ncomp, int i0, int cnt, double* out, hipStream_t s);
int qxk_pairm_sym(int n, double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix, hipStream_t s);
int qxk_pairm_expand(int n, const double* M, long long ld, long long slice, int nslice, const QxPairIndex* ix,
                     const int* index, const int* fn, double* out, hipStream_t s);
int qxk_pairm_ao(const QxShellsDev* sh, const QxPairIndex* ix, const int* fn, double* M, long long ld, long long slice,
                 int nslice, hipStream_t s);
int qxk_oei_deriv(const QxShellsDev* sh, double* dS, double* dT, double* dV, hipStream_t s);
}
