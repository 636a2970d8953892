// Host runtime of the MI355X ERI library: context set-up (normalisation,
// Boys table, shell pairs, Schwarz screening on the device, quartet lists)
// and the C-ABI entry points declared in include/quax_amd.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <numeric>
#include <stdexcept>
#include <string>
#include <vector>

#include "quax_amd.h"
#include "qx_oei.h"
#include "qx_runtime.h"
#include "qx_rys.h"
#include "qx_classes.inc"  // generated; in the build's generated-source directory

static_assert(QX_GEN_LMAX == QX_LMAX_SUPPORTED, "generated kernels and runtime disagree on lmax");
static_assert(QX_NUM_CLASSES == QX_NUM_CLASSES_MAX, "profile slot layout");

namespace {

struct QxError {
  int code;
  std::string msg;
};

#define QX_HIP(call)                                                                            \
  do {                                                                                          \
    hipError_t e_ = (call);                                                                     \
    if (e_ != hipSuccess)                                                                       \
      throw QxError{e_ == hipErrorOutOfMemory ? QX_ENOMEM : QX_EHIP,                            \
                    std::string(#call) + ": " + hipGetErrorString(e_)};                         \
  } while (0)

#define QX_REQUIRE(cond, code, msg) \
  do {                              \
    if (!(cond)) throw QxError{code, msg}; \
  } while (0)

int ncart(int l) { return (l + 1) * (l + 2) / 2; }
int nsph(int l, int pure) { return (pure && l >= 2) ? 2 * l + 1 : ncart(l); }
int pair_class(int la, int lb) { return la * (la + 1) / 2 + lb; }

template <class T>
T* dalloc(qx_ctx* c, size_t n) {
  void* p = nullptr;
  QX_HIP(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)));
  c->allocs.push_back(p);
  return static_cast<T*>(p);
}

template <class T>
T* dupload(qx_ctx* c, const std::vector<T>& v) {
  T* p = dalloc<T>(c, v.size());
  if (!v.empty()) QX_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return p;
}

// scoped temporary device buffer
struct DevBuf {
  void* p = nullptr;
  explicit DevBuf(void* owned) : p(owned) {}
  explicit DevBuf(size_t bytes) { QX_HIP(hipMalloc(&p, std::max<size_t>(bytes, 8))); }
  ~DevBuf() { if (p) (void)hipFree(p); }
  double* d() const { return static_cast<double*>(p); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
};

double dfact(int n) {
  double r = 1.0;
  for (int k = n; k > 1; k -= 2) r *= k;
  return r;
}

// Libint Shell::renorm convention: x^l normalisation of each primitive,
// then the contraction rescaled to unit self-overlap.
void normalize_shell(int l, int np, const double* a, const double* cin, double* cout) {
  const double pi32 = std::pow(M_PI, 1.5);
  for (int p = 0; p < np; ++p) {
    const double two_a = 2.0 * a[p];
    cout[p] = cin[p] * std::sqrt(std::pow(2.0, l) * std::pow(two_a, l + 1.5) / (pi32 * dfact(2 * l - 1)));
  }
  double s = 0.0;
  for (int p = 0; p < np; ++p)
    for (int q = 0; q < np; ++q)
      s += dfact(2 * l - 1) * pi32 * cout[p] * cout[q] / (std::pow(2.0, l) * std::pow(a[p] + a[q], l + 1.5));
  const double f = 1.0 / std::sqrt(s);
  for (int p = 0; p < np; ++p) cout[p] *= f;
}

// Boys table rows F_0..F_{NM-1}(g/INV_H): series at the top order in long
// double, F_m(T) = exp(-T) sum_k (2T)^k / ((2m+1)(2m+3)...(2m+2k+1)),
// then downward recursion F_{m-1} = (2T F_m + exp(-T)) / (2m-1).
std::vector<double> boys_table() {
  std::vector<double> tab((size_t)QX_BOYS_NPTS * QX_BOYS_NM);
  for (int g = 0; g < QX_BOYS_NPTS; ++g) {
    const long double T = g / (long double)QX_BOYS_INV_H;
    const int M = QX_BOYS_NM - 1;
    long double term = 1.0L / (2 * M + 1), sum = term;
    for (int k = 1; k < 4000; ++k) {
      term *= 2.0L * T / (2 * M + 2 * k + 1);
      sum += term;
      if (term < 1e-26L * sum) break;
    }
    const long double et = expl(-T);
    long double f = et * sum;
    tab[(size_t)g * QX_BOYS_NM + M] = (double)f;
    for (int m = M; m > 0; --m) {
      f = (2.0L * T * f + et) / (2 * m - 1);
      tab[(size_t)g * QX_BOYS_NM + m - 1] = (double)f;
    }
  }
  return tab;
}

// real solid harmonics for l = 2 in terms of x^l-normalised Cartesians
// (xx, xy, xz, yy, yz, zz), rows m = -2..2, unit-normalised.
const double kSph2[5 * 6] = {
    0, 1.7320508075688772, 0, 0, 0, 0,                   // m=-2: sqrt3 xy
    0, 0, 0, 0, 1.7320508075688772, 0,                   // m=-1: sqrt3 yz
    -0.5, 0, 0, -0.5, 0, 1.0,                            // m= 0: z^2 - (x^2+y^2)/2
    0, 0, 1.7320508075688772, 0, 0, 0,                   // m=+1: sqrt3 xz
    0.8660254037844386, 0, 0, -0.8660254037844386, 0, 0  // m=+2: sqrt3/2 (x^2-y^2)
};

struct PairRec {
  int a, b;        // oriented shells (l[a] >= l[b])
  int s1, s2;      // reference order (s1 >= s2)
  int cls;
  double Q;
};

void build_pair_arrays(qx_ctx* c, const std::vector<PairRec>& P, QxPairsDev& pr, QxPrimPairsDev& pp, int& npseudo,
                       std::vector<int>* h_first, std::vector<int>* h_n) {
  const int np = (int)P.size();
  std::vector<double> Ax(np), Ay(np), Az(np), ABx(np), ABy(np), ABz(np);
  std::vector<int> sa(np), sb(np), bfa(np), bfb(np), ata(np), atb(np), first(np), cnt(np);
  std::vector<int> ppair;
  std::vector<double> p_, Px, Py, Pz, K, a2, b2;
  for (int i = 0; i < np; ++i) {
    const int a = P[i].a, b = P[i].b;
    const double* A = &c->xyz[3 * c->atom[a]];
    const double* B = &c->xyz[3 * c->atom[b]];
    Ax[i] = A[0]; Ay[i] = A[1]; Az[i] = A[2];
    ABx[i] = A[0] - B[0]; ABy[i] = A[1] - B[1]; ABz[i] = A[2] - B[2];
    sa[i] = a; sb[i] = b;
    bfa[i] = c->bfc[a]; bfb[i] = c->bfc[b];
    ata[i] = c->atom[a]; atb[i] = c->atom[b];
    first[i] = (int)ppair.size();
    const double AB2 = ABx[i] * ABx[i] + ABy[i] * ABy[i] + ABz[i] * ABz[i];
    for (int ia = c->poff[a]; ia < c->poff[a] + c->nprim[a]; ++ia)
      for (int ib = c->poff[b]; ib < c->poff[b] + c->nprim[b]; ++ib) {
        const double al = c->exps[ia], be = c->exps[ib], p = al + be;
        ppair.push_back(i);
        p_.push_back(p);
        Px.push_back((al * A[0] + be * B[0]) / p);
        Py.push_back((al * A[1] + be * B[1]) / p);
        Pz.push_back((al * A[2] + be * B[2]) / p);
        K.push_back(c->coefs[ia] * c->coefs[ib] * std::exp(-al * be / p * AB2));
        a2.push_back(2 * al);
        b2.push_back(2 * be);
      }
    cnt[i] = (int)ppair.size() - first[i];
  }
  npseudo = (int)ppair.size();
  pr.Ax = dupload(c, Ax); pr.Ay = dupload(c, Ay); pr.Az = dupload(c, Az);
  pr.ABx = dupload(c, ABx); pr.ABy = dupload(c, ABy); pr.ABz = dupload(c, ABz);
  pr.sa = dupload(c, sa); pr.sb = dupload(c, sb);
  pr.bfa = dupload(c, bfa); pr.bfb = dupload(c, bfb);
  pr.atom_a = dupload(c, ata); pr.atom_b = dupload(c, atb);
  pr.pp_first = dupload(c, first); pr.pp_n = dupload(c, cnt);
  pp.pair = dupload(c, ppair);
  pp.p = dupload(c, p_); pp.Px = dupload(c, Px); pp.Py = dupload(c, Py); pp.Pz = dupload(c, Pz);
  pp.K = dupload(c, K); pp.a2 = dupload(c, a2); pp.b2 = dupload(c, b2);
  if (h_first) *h_first = first;
  if (h_n) *h_n = cnt;
}

hipEvent_t take_event(qx_ctx* c) {
  if (!c->event_pool.empty()) {
    hipEvent_t e = c->event_pool.back();
    c->event_pool.pop_back();
    return e;
  }
  hipEvent_t e;
  QX_HIP(hipEventCreate(&e));
  return e;
}

// Runs one kernel launch, bracketed by HIP events on its stream when
// profiling is on (and the pass may use events: `timed`).
template <class F>
int timed_launch(qx_ctx* c, int slot, long long pq, hipStream_t s, F&& launch, bool timed = true) {
  if (!timed || !c->profiling || pq <= 0) return launch();
  hipEvent_t a = take_event(c), b = take_event(c);
  QX_HIP(hipEventRecord(a, s));
  const int rc = launch();
  QX_HIP(hipEventRecord(b, s));
  c->prof_pending.push_back({slot, a, b});
  c->prof_launches[slot] += 1;
  c->prof_pq[slot] += pq;
  return rc;
}

int launch_eri(qx_ctx* c, const QxWorkDev& w, int cls, const QxEpiDev& e, int fp32, hipStream_t s,
               const QxPairsDev& pr, const QxPrimPairsDev& pp, const QxPairM* pm, const QxKList* kl) {
  QxArgs a;
  a.pr = pr; a.pp = pp; a.w = w; a.e = e; a.boys = c->d_boys;
  QxLaunch L{fp32, s, 0, pm, kl};
  const QxClassEntry& ent = qx_class_table[cls];
  return timed_launch(c, QX_SLOT_ERI(cls, fp32 ? 1 : 0), w.nquart, s, [&] { return ent.eri(&a, &L); });
}

// One kernel launch of a pass, with its estimated cost (flops).
struct Launch {
  double cost;
  std::function<int(hipStream_t)> go;
};

void ensure_side_streams(qx_ctx* c) {
  const int want = std::max(0, c->nstreams - 1);
  while ((int)c->side.size() < want) {
    hipStream_t t;
    QX_HIP(hipStreamCreateWithFlags(&t, hipStreamNonBlocking));
    c->side.push_back(t);
  }
  while ((int)c->fork_ev.size() < want + 1) {
    hipEvent_t e;
    QX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    c->fork_ev.push_back(e);
  }
}

void check_launch(int rc, const char* what);

// Runs the independent launches of one pass.  With several streams the
// costliest go first, each to the least-loaded stream; the side streams wait
// for the caller's stream before starting and the caller's stream waits for
// all of them at the end, so the pass is ordered on `s` like one kernel.
// With profiling on, each kernel's HIP events sit on the stream it runs on:
// concurrent kernels are timed in place (one stream times each alone).
//
// side = false keeps the pass on the caller's stream (callers that may not use
// events or other streams).  Scratch: each hardware queue grows its own to the
// largest per-lane size it has run, and growing a side stream's queue past
// ~8 KB per lane once the process holds scratch on its other queues has been
// refused by the HSA runtime (HSA_STATUS_ERROR_OUT_OF_RESOURCES); the build
// keeps every kernel that runs here under 6 KB.
void run_launches(qx_ctx* c, std::vector<Launch>& v, hipStream_t s, const char* what, bool side) {
  // two small launches cost less in turn than the events of a fork (H2's
  // directional J/K 47 us against 71)
  double cost = 0.0;
  for (const auto& x : v) cost += x.cost;
  if (v.size() <= 2 && cost < 1e8) side = false;
  const int ns = side ? std::max(1, std::min<int>(c->nstreams, (int)v.size())) : 1;
  if (ns == 1) {
    for (auto& x : v) check_launch(x.go(s), what);
    return;
  }
  ensure_side_streams(c);
  std::stable_sort(v.begin(), v.end(), [](const Launch& a, const Launch& b) { return a.cost > b.cost; });
  QX_HIP(hipEventRecord(c->fork_ev[0], s));
  for (int k = 0; k < ns - 1; ++k) QX_HIP(hipStreamWaitEvent(c->side[k], c->fork_ev[0], 0));
  std::vector<double> load(ns, 0.0);
  int rc = 0;
  std::exception_ptr thrown;
  for (auto& x : v) {
    const int k = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[k] += x.cost;
    try {
      rc = x.go(k == 0 ? s : c->side[k - 1]);
    } catch (...) {
      thrown = std::current_exception();
    }
    if (rc != 0 || thrown) break;
  }
  // join even after a failed or throwing launch, so the caller's stream
  // never runs ahead of work already queued on the side streams
  hipError_t join_err = hipSuccess;
  for (int k = 0; k < ns - 1; ++k) {
    hipError_t e = hipEventRecord(c->fork_ev[k + 1], c->side[k]);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, c->fork_ev[k + 1], 0);
    if (e != hipSuccess && join_err == hipSuccess) join_err = e;
  }
  if (thrown) std::rethrow_exception(thrown);
  check_launch(rc, what);
  QX_HIP(join_err);
}

void check_launch(int rc, const char* what) {
  if (rc == -1) throw QxError{QX_EUNSUPPORTED, std::string(what) + ": kernel variant not built"};
  if (rc != 0) throw QxError{QX_EHIP, std::string(what) + ": " + hipGetErrorString((hipError_t)rc)};
}

int class_index(int X, int Y) { return X * (X + 1) / 2 + Y; }

// Positions [ss, se) of fragment f within the class list that starts at
// sorted pair ko and holds kn pairs (sorted by fragment, then Schwarz value).
void frag_segment(const qx_ctx* c, int ko, int kn, int f, int& ss, int& se) {
  const int* fr = c->h_pair_frag.data() + ko;
  ss = (int)(std::lower_bound(fr, fr + kn, f) - fr);
  se = (int)(std::upper_bound(fr, fr + kn, f) - fr);
}

// Admissible kets of every bra pair of class X in class Y: positions
// [first, first + count) of Y's list, i.e. the bra's fragment and
// Q_bra Q_ket >= bound, a prefix of the segment, which is sorted by descending
// Q.  The bras of a fragment are too, so the prefix only shrinks from one to
// the next.  (`canonical`: j <= i when X == Y.)
std::vector<QxRange> ket_windows(const qx_ctx* c, int X, int Y, double bound, bool canonical = true) {
  const int bo = c->class_pair_off[X], bn = c->class_pair_cnt[X];
  const int ko = c->class_pair_off[Y], kn = c->class_pair_cnt[Y];
  std::vector<QxRange> w(bn);
  int ss = 0, end = 0;
  for (int i = 0; i < bn; ++i) {
    if (i == 0 || c->h_pair_frag[bo + i] != c->h_pair_frag[bo + i - 1])
      frag_segment(c, ko, kn, c->h_pair_frag[bo + i], ss, end);
    while (end > ss && !(c->h_pair_Q[bo + i] * c->h_pair_Q[ko + end - 1] >= bound)) --end;
    int kc = end - ss;
    if (X == Y && canonical) kc = std::max(0, std::min(kc, i - ss + 1));
    w[i] = {ss, kc};
  }
  return w;
}

// Pseudo kets of each class that every pair (any order of the two classes)
// meets with Q_P Q_ket >= bound: the J kernels' ranges, [Y * npairs + pair].
std::vector<QxRange> pseudo_ranges(const qx_ctx* c, double bound) {
  std::vector<QxRange> r((size_t)6 * c->npairs, QxRange{0, 0});
  for (int X = 0; X < 6; ++X)
    for (int Y = 0; Y < 6; ++Y) {
      const int ko = c->class_pair_off[Y];
      const auto w = ket_windows(c, X, Y, bound, false);
      for (size_t i = 0; i < w.size(); ++i) {
        if (w[i].count <= 0) continue;
        const int first = ko + w[i].first, last = first + w[i].count - 1;
        r[(size_t)Y * c->npairs + c->class_pair_off[X] + i] = {c->h_pp_first[first],
                                                               c->h_pp_first[last] + c->h_pp_n[last] - c->h_pp_first[first]};
      }
    }
  return r;
}

// Work matrices of qx_jk_build_noalloc in the file-scope array `scratch`.
#define QX_NOALLOC_DOUBLES (3ull << 20)
// Doubles of it that a context is charged with (the documented limit; a
// spherical pass uses three of its five matrices).
size_t noalloc_doubles(const qx_ctx* c) { return (size_t)(c->pure ? 5 : 2) * c->ncart * c->ncart; }

// Hermite layout and J ranges.
void setup_jk(qx_ctx* c) {
  static const int order[6] = {0, 1, 2, 2, 3, 4};
  QxJList& jl = c->jlist;
  jl.npairs = c->npairs;
  long long at = 0;
  int u = 0;
  for (int X = 0; X < 6; ++X) {
    const int cnt = c->class_pair_cnt[X], off = c->class_pair_off[X];
    const int nu = cnt ? c->h_pp_first[off + cnt - 1] + c->h_pp_n[off + cnt - 1] - c->h_pp_first[off] : 0;
    jl.uoff[X] = u;
    jl.hoff[X] = (int)at;
    u += nu;
    at += (long long)nu * qx_nherm(order[X]);
  }
  jl.uoff[6] = u;
  QX_REQUIRE(at <= 0x7fffffff, QX_EUNSUPPORTED, "too many primitive pairs");
  c->nherm = at;
  c->d_range = dupload(c, pseudo_ranges(c, c->tol * c->tol));
  c->d_herm = dalloc<double>(c, (size_t)4 * at);
  jl.range = c->d_range;
  jl.H = c->d_herm;
  jl.P = c->d_herm + at;
  jl.Hd = c->d_herm + 2 * at;
  jl.Pd = c->d_herm + 3 * at;
  // the allocation-free pass has its own, as it may run beside another pass
  if (noalloc_doubles(c) <= QX_NOALLOC_DOUBLES) c->d_herm_own = dalloc<double>(c, (size_t)2 * at);
}

void schwarz_and_lists(qx_ctx* c) {
  const int ns = c->nshell;
  c->d_rys = dalloc<double>(c, QX_RYS_DOUBLES);
  QX_HIP(hipMemcpy(c->d_rys, qxk_rys_host(), QX_RYS_DOUBLES * sizeof(double), hipMemcpyHostToDevice));
  // ---- every shell pair, class-sorted, for the Schwarz pass
  std::vector<PairRec> all;
  for (int s1 = 0; s1 < ns; ++s1)
    for (int s2 = 0; s2 <= s1; ++s2) {
      if (c->frag[c->atom[s1]] != c->frag[c->atom[s2]]) continue;  // pairs never span fragments
      PairRec r;
      r.s1 = s1; r.s2 = s2;
      if (c->l[s1] >= c->l[s2]) { r.a = s1; r.b = s2; } else { r.a = s2; r.b = s1; }
      r.cls = pair_class(c->l[r.a], c->l[r.b]);
      r.Q = 0.0;
      all.push_back(r);
    }
  std::stable_sort(all.begin(), all.end(), [](const PairRec& x, const PairRec& y) { return x.cls < y.cls; });
  QxPairsDev pr_all{};
  QxPrimPairsDev pp_all{};
  int np_all = 0;
  const size_t alloc_mark = c->allocs.size();
  std::vector<int> first, cnt;
  build_pair_arrays(c, all, pr_all, pp_all, np_all, &first, &cnt);
  const int npair_all = (int)all.size();
  DevBuf diag((size_t)npair_all * QX_PAIR_STRIDE * sizeof(double));
  check_launch(qxk_fill(diag.d(), (long long)npair_all * QX_PAIR_STRIDE, 0.0, 0), "fill");
  // diagonal lists per pair class: bra = pseudo pairs of the class, kets =
  // the pseudo pairs of the same contracted pair
  const int nclass = pair_class(QX_LMAX_SUPPORTED, QX_LMAX_SUPPORTED) + 1;
  std::vector<std::vector<long long>> pre(nclass);
  std::vector<QxWorkDev> wl(nclass);
  std::vector<DevBuf*> bufs;
  for (int X = 0; X < nclass; ++X) {
    int lo = -1, hi = -1;
    for (int i = 0; i < npair_all; ++i)
      if (all[i].cls == X) { if (lo < 0) lo = i; hi = i + 1; }
    if (lo < 0) continue;
    const int u0 = first[lo], u1 = first[hi - 1] + cnt[hi - 1];
    std::vector<long long> p(u1 - u0 + 1, 0);
    int idx = 0;
    for (int i = lo; i < hi; ++i)
      for (int k = 0; k < cnt[i]; ++k, ++idx) p[idx + 1] = p[idx] + cnt[i];
    DevBuf* b = new DevBuf(p.size() * sizeof(long long));
    bufs.push_back(b);
    QX_HIP(hipMemcpy(b->p, p.data(), p.size() * sizeof(long long), hipMemcpyHostToDevice));
    QxWorkDev w{};
    w.bra_off = u0; w.nbra = u1 - u0; w.ket_off = 0; w.nket = 0;
    w.prefix = static_cast<const long long*>(b->p);
    w.nquart = p.back(); w.store_base = 0; w.diag = 1;
    QxEpiDev e{};
    e.epi = QX_EPI_SCHWARZ; e.out = diag.d(); e.nbf = c->ncart; e.natom = c->natom; e.coord = -1;
    QxKList kl{};
    kl.bra0 = lo; kl.nbra = hi - lo; kl.rys = c->d_rys;
    for (int i = lo; i < hi; ++i) kl.ketprim = std::max(kl.ketprim, cnt[i]);
    int rc = launch_eri(c, w, class_index(X, X), e, 0, 0, pr_all, pp_all, nullptr, &kl);
    if (rc != 0) {
      for (auto* q : bufs) delete q;
      check_launch(rc, "schwarz");
    }
  }
  hipError_t se = hipDeviceSynchronize();
  for (auto* q : bufs) delete q;
  QX_HIP(se);
  std::vector<double> hd((size_t)npair_all * QX_PAIR_STRIDE);
  QX_HIP(hipMemcpy(hd.data(), diag.p, hd.size() * sizeof(double), hipMemcpyDeviceToHost));
  c->Q.assign((size_t)ns * ns, 0.0);
  double maxq = 0.0;
  for (int i = 0; i < npair_all; ++i) {
    const int na = ncart(c->l[all[i].a]), nb = ncart(c->l[all[i].b]);
    double m = 0.0;
    for (int k = 0; k < na * nb; ++k) m = std::max(m, std::fabs(hd[(size_t)i * QX_PAIR_STRIDE + k]));
    all[i].Q = m;
    c->Q[(size_t)all[i].s1 * ns + all[i].s2] = c->Q[(size_t)all[i].s2 * ns + all[i].s1] = m;
    maxq = std::max(maxq, m);
  }
  // release the all-pairs arrays
  while (c->allocs.size() > alloc_mark) {
    (void)hipFree(c->allocs.back());
    c->allocs.pop_back();
  }
  // ---- screening (libint_interface.cc:215-225)
  const double tol2 = c->tol * c->tol;
  const double cut = tol2 / maxq;
  c->ref_pairs.clear();
  for (int s1 = 0; s1 < ns; ++s1)
    for (int s2 = 0; s2 <= s1; ++s2)
      if (c->Q[(size_t)s1 * ns + s2] >= cut) { c->ref_pairs.push_back(s1); c->ref_pairs.push_back(s2); }
  std::vector<PairRec> scr;
  for (auto& r : all)
    if (r.Q >= cut) scr.push_back(r);
  std::sort(scr.begin(), scr.end(), [c](const PairRec& x, const PairRec& y) {
    if (x.cls != y.cls) return x.cls < y.cls;
    const int fx = c->frag[c->atom[x.a]], fy = c->frag[c->atom[y.a]];
    if (fx != fy) return fx < fy;
    if (x.Q != y.Q) return x.Q > y.Q;
    if (x.s1 != y.s1) return x.s1 < y.s1;
    return x.s2 < y.s2;
  });
  build_pair_arrays(c, scr, c->pr, c->pp, c->npseudo, &c->h_pp_first, &c->h_pp_n);
  c->class_prims.assign(6, 1);
  for (size_t i = 0; i < scr.size(); ++i) c->class_prims[scr[i].cls] = std::max(c->class_prims[scr[i].cls], c->h_pp_n[i]);
  c->npairs = (int)scr.size();
  c->h_pair_sa.resize(c->npairs); c->h_pair_sb.resize(c->npairs);
  c->h_pair_class.resize(c->npairs); c->h_pair_Q.resize(c->npairs); c->h_pair_frag.resize(c->npairs);
  for (int i = 0; i < c->npairs; ++i) {
    c->h_pair_sa[i] = scr[i].a; c->h_pair_sb[i] = scr[i].b;
    c->h_pair_class[i] = scr[i].cls; c->h_pair_Q[i] = scr[i].Q;
    c->h_pair_frag[i] = c->frag[c->atom[scr[i].a]];
  }
  c->class_pair_off.assign(nclass, 0); c->class_pair_cnt.assign(nclass, 0);
  for (int i = c->npairs - 1; i >= 0; --i) c->class_pair_off[scr[i].cls] = i;
  for (int i = 0; i < c->npairs; ++i) c->class_pair_cnt[scr[i].cls]++;
  // ---- quartet lists
  c->work.clear();
  c->nq_class.assign(QX_NUM_CLASSES, 0);
  c->ndq_class.assign(QX_NUM_CLASSES, 0);
  // positions (within their class) of pairs whose two shells sit on one atom,
  // per (class, atom), to count single-atom quartets
  std::vector<std::vector<std::vector<int>>> intra(nclass, std::vector<std::vector<int>>(c->natom));
  for (int X = 0; X < nclass; ++X)
    for (int i = 0; i < c->class_pair_cnt[X]; ++i) {
      const int P = c->class_pair_off[X] + i;
      const int A = c->atom[c->h_pair_sa[P]];
      if (A == c->atom[c->h_pair_sb[P]]) intra[X][A].push_back(i);
    }
  std::vector<long long> allpre;
  std::vector<int> allkst;  // per bra pseudo pair: first ket (fragmented contexts)
  std::vector<long long> allcpre;  // the same over contracted pairs
  std::vector<int> allckst;
  std::vector<long long> kst_off;
  c->nquart_total = 0; c->npq_total = 0; c->store_total = 0;
  for (int X = 0; X < nclass; ++X) {
    for (int Y = 0; Y <= X; ++Y) {
      const int bo = c->class_pair_off[X], bn = c->class_pair_cnt[X];
      const int ko = c->class_pair_off[Y], kn = c->class_pair_cnt[Y];
      if (bn == 0 || kn == 0) continue;
      // cumulative pseudo counts over the ket class
      std::vector<long long> kcum(kn + 1, 0);
      for (int j = 0; j < kn; ++j) kcum[j + 1] = kcum[j] + c->h_pp_n[ko + j];
      QxWorkHost wh{};
      wh.cls = class_index(X, Y);
      wh.bra_class = X; wh.ket_class = Y;
      wh.prefix_off = (long long)allpre.size();
      wh.cprefix_off = (long long)allcpre.size();
      allcpre.push_back(0);
      const int u0 = c->h_pp_first[bo];
      const int u1 = c->h_pp_first[bo + bn - 1] + c->h_pp_n[bo + bn - 1];
      allpre.push_back(0);
      kst_off.push_back((long long)allkst.size());
      long long run = 0, ncq = 0;
      const auto window = ket_windows(c, X, Y, tol2);
      for (int i = 0; i < bn; ++i) {
        const int ss = window[i].first, kc = window[i].count;
        ncq += kc;
        wh.maxket = std::max(wh.maxket, kc);
        allcpre.push_back(ncq);
        allckst.push_back(ss);
        {
          const int P = bo + i;
          const int A = c->atom[c->h_pair_sa[P]];
          long long single = 0;
          if (A == c->atom[c->h_pair_sb[P]]) {
            const auto& v = intra[Y][A];
            single = (std::lower_bound(v.begin(), v.end(), ss + kc) - v.begin()) -
                     (std::lower_bound(v.begin(), v.end(), ss) - v.begin());
          }
          c->ndq_class[class_index(X, Y)] += kc - single;
        }
        for (int k = 0; k < c->h_pp_n[bo + i]; ++k) {
          run += kcum[ss + kc] - kcum[ss];
          allpre.push_back(run);
          allkst.push_back((int)kcum[ss]);
        }
      }
      wh.w.bra_off = u0; wh.w.nbra = u1 - u0;
      wh.w.ket_off = c->h_pp_first[ko];
      wh.w.nket = (int)kcum[kn];
      wh.w.nquart = run;
      wh.w.diag = 0;
      wh.ncq = ncq;
      wh.prims = (int)std::max((run + ncq - 1) / std::max(ncq, 1LL), 1LL);
      allckst.push_back(0);  // one entry per prefix entry
      wh.w.store_base = c->store_total;
      const int N = ncart(c->l[c->h_pair_sa[bo]]) * ncart(c->l[c->h_pair_sb[bo]]) *
                    ncart(c->l[c->h_pair_sa[ko]]) * ncart(c->l[c->h_pair_sb[ko]]);
      c->store_total += run * N;
      c->nquart_total += ncq;
      c->nq_class[class_index(X, Y)] += ncq;
      c->npq_total += run;
      if (run > 0) {
        c->work.push_back(wh);
      } else {
        allpre.resize(wh.prefix_off);
        allcpre.resize(wh.cprefix_off);
        allckst.resize(wh.cprefix_off);
        allkst.resize(kst_off.back());
        kst_off.pop_back();
      }
    }
  }
  c->d_prefix = dupload(c, allpre);
  c->d_cprefix = dupload(c, allcpre);
  if (c->fragmented) {
    c->d_kstart = dupload(c, allkst);
    c->d_ckstart = dupload(c, allckst);
    c->d_pair_frag = dupload(c, c->h_pair_frag);
    // Cartesian function range of each fragment id (all kets of a bra pair
    // lie in its fragment, so a block's K' rows span at most this range)
    int fmax = 0;
    for (int f : c->frag) fmax = std::max(fmax, f);
    std::vector<int> lo(fmax + 1, INT32_MAX), hi(fmax + 1, -1);
    for (int sh = 0; sh < c->nshell; ++sh) {
      const int f = c->frag[c->atom[sh]];
      lo[f] = std::min(lo[f], c->bfc[sh]);
      hi[f] = std::max(hi[f], c->bfc[sh] + ncart(c->l[sh]));
    }
    c->kcols = 0;
    for (int f = 0; f <= fmax; ++f) {
      if (hi[f] < 0) lo[f] = 0;
      else c->kcols = std::max(c->kcols, hi[f] - lo[f]);
    }
    c->d_frag_col0 = dupload(c, lo);
    // atom window of each fragment id: lowest atom, atoms up to the highest
    std::vector<int> win(2 * (size_t)(fmax + 1), 0);
    for (int at = 0; at < c->natom; ++at) {
      int* w = &win[2 * (size_t)c->frag[at]];
      if (w[1] == 0) w[0] = at;
      w[1] = at - w[0] + 1;
    }
    c->d_frag_atoms = dupload(c, win);
  }
  c->h_prefix = allpre;
  c->h_cprefix = allcpre;
  c->h_kstart = allkst;
  c->h_kstart_off = kst_off;
  c->h_ppair.assign(c->npseudo, 0);
  for (int i = 0; i < c->npairs; ++i)
    for (int k = 0; k < c->h_pp_n[i]; ++k) c->h_ppair[c->h_pp_first[i] + k] = i;
  for (size_t k = 0; k < c->work.size(); ++k) {
    auto& wh = c->work[k];
    wh.w.prefix = c->d_prefix + wh.prefix_off;
    wh.w.kstart = c->fragmented ? c->d_kstart + kst_off[k] : nullptr;
  }
}

#define QX_JK_ROWS_NMAX 2048

// K' rows of a J/K pass in LDS (each class kernel still decides whether its
// rows fit): over the bra fragment's function range in a fragmented context,
// over all functions otherwise; none when that width exceeds
// QX_JK_ROWS_NMAX, where zeroing and scanning a block's rows would cost more
// than its quartets.
static void set_krows(const qx_ctx* c, QxEpiDev& e) {
  const int width = c->fragmented ? c->kcols : c->ncart;
  e.krows = width <= QX_JK_ROWS_NMAX ? 1 : 0;
  if (c->fragmented) {
    e.kcols = c->kcols;
    e.frag_col0 = c->d_frag_col0;
    e.pair_frag = c->d_pair_frag;
  }
}

// Copies of the 3N gradient accumulators of an adjoint-gradient pass,
// cleared on stream s (the pass's blocks flush into copy block % copies; the
// runtime adds the copies to the caller's gradient after the pass).
#define QX_GRAD_COPIES 64
static double* begin_grad_copies(qx_ctx* c, hipStream_t s) {
  const long long n = (long long)QX_GRAD_COPIES * 3 * c->natom;
  if (!c->gcopies) c->gcopies = dalloc<double>(c, (size_t)n);
  check_launch(qxk_fill(c->gcopies, n, 0.0, s), "fill");
  return c->gcopies;
}

// Orders a pass on stream s after the previous user of the context's
// workspaces.
void order_ws(qx_ctx* c, hipStream_t s) {
  if (!c->ws_ev) QX_HIP(hipEventCreateWithFlags(&c->ws_ev, hipEventDisableTiming));
  if (c->ws_used && !c->capturing) QX_HIP(hipStreamWaitEvent(s, c->ws_ev, 0));
}

// Work matrices of a J/K or gradient pass on stream s (see qx_ctx::ws).
double* begin_ws(qx_ctx* c, hipStream_t s) {
  if (!c->ws) c->ws = dalloc<double>(c, (size_t)5 * c->ncart * c->ncart);
  order_ws(c, s);
  return c->ws;
}

void end_ws(qx_ctx* c, hipStream_t s) {
  if (c->capturing) return;
  QX_HIP(hipEventRecord(c->ws_ev, s));
  c->ws_used = true;
}

// Mixed precision: for every quartet list, the number of FP64 kets of each
// bra pair at a Schwarz-bound threshold.  Kets of each bra pair are sorted by
// descending Q, so for bra i the FP64 kets (Q_i Q_j >= thr^2) are a prefix of
// its admissible kets; a launch then takes either part of every row (kl.sel).
void build_split(qx_ctx* c, double thr) {
  auto& S = c->split;
  if (S.thr == thr) return;
  QX_HIP(hipDeviceSynchronize());  // no kernel may still read the old counts
  for (int* p : {S.d_ck64, S.d_range64})
    if (p) (void)hipFree(p);
  S = qx_ctx::Split{};
  const double tol2 = c->tol * c->tol, thr2 = thr * thr;
  std::vector<int> ck(c->h_cprefix.size(), 0);  // per list, per bra pair
  for (const auto& wh : c->work) {
    const int X = wh.bra_class, Y = wh.ket_class;
    const int bo = c->class_pair_off[X], bn = c->class_pair_cnt[X];
    const int ko = c->class_pair_off[Y], kn = c->class_pair_cnt[Y];
    std::vector<long long> kcum(kn + 1, 0);
    for (int j = 0; j < kn; ++j) kcum[j + 1] = kcum[j] + c->h_pp_n[ko + j];
    long long p64 = 0, p32 = 0, q64 = 0, q32 = 0;
    const auto all = ket_windows(c, X, Y, tol2), fp64 = ket_windows(c, X, Y, thr2);
    for (int i = 0; i < bn; ++i) {
      const int ss = all[i].first, kc = all[i].count, k64 = std::min(kc, fp64[i].count);
      q64 += k64;
      q32 += kc - k64;
      ck[wh.cprefix_off + i] = k64;
      const long long r64 = kcum[ss + k64] - kcum[ss], rall = kcum[ss + kc] - kcum[ss];
      for (int k = 0; k < c->h_pp_n[bo + i]; ++k) {
        p64 += r64;
        p32 += rall - r64;
      }
    }
    if (p64 + p32 != wh.w.nquart) throw QxError{QX_EHIP, "mixed-precision split lost quartets"};
    S.pq64.push_back(p64); S.pq32.push_back(p32);
    S.cq64.push_back(q64); S.cq32.push_back(q32);
  }
  const auto rall = pseudo_ranges(c, tol2), rthr = pseudo_ranges(c, thr2);
  std::vector<int> r64(rall.size());
  for (size_t i = 0; i < r64.size(); ++i) r64[i] = std::min(rall[i].count, rthr[i].count);
  QX_HIP(hipMalloc(&S.d_ck64, std::max<size_t>(ck.size(), 1) * sizeof(int)));
  if (!ck.empty()) QX_HIP(hipMemcpy(S.d_ck64, ck.data(), ck.size() * sizeof(int), hipMemcpyHostToDevice));
  QX_HIP(hipMalloc(&S.d_range64, std::max<size_t>(r64.size(), 1) * sizeof(int)));
  if (!r64.empty()) QX_HIP(hipMemcpy(S.d_range64, r64.data(), r64.size() * sizeof(int), hipMemcpyHostToDevice));
  S.thr = thr;
}

void setup_shell_tables(qx_ctx* c) {
  QxShellsDev& s = c->shells;
  s.nshell = c->nshell; s.natom = c->natom; s.ncart = c->ncart; s.nbf = c->nbf; s.pure = c->pure;
  s.l = dupload(c, c->l); s.atom = dupload(c, c->atom); s.nprim = dupload(c, c->nprim);
  s.poff = dupload(c, c->poff); s.bfc = dupload(c, c->bfc); s.bfs = dupload(c, c->bfs);
  s.exps = dupload(c, c->exps); s.coefs = dupload(c, c->coefs);
  s.xyz = dupload(c, c->xyz); s.Z = dupload(c, c->Z);
  std::vector<int> fs, fc, as;
  for (int sh = 0; sh < c->nshell; ++sh) {
    const int l = c->l[sh];
    for (int i = 0; i <= l; ++i)
      for (int j = 0; j <= i; ++j) {
        fs.push_back(sh);
        fc.push_back(((l - i) << 16) | ((i - j) << 8) | j);
      }
    for (int k = 0; k < nsph(l, c->pure); ++k) as.push_back(sh);
  }
  // shells grouped by angular momentum (one-electron pair classes)
  std::vector<int> by_l;
  for (int l = 0; l <= QX_LMAX_SUPPORTED; ++l) {
    c->l_off[l] = (int)by_l.size();
    for (int sh = 0; sh < c->nshell; ++sh)
      if (c->l[sh] == l) by_l.push_back(sh);
  }
  c->l_off[QX_LMAX_SUPPORTED + 1] = (int)by_l.size();
  c->d_shell_by_l = dupload(c, by_l);
  s.f_shell = dupload(c, fs); s.f_comp = dupload(c, fc); s.ao_shell = dupload(c, as);
  // transform blocks: identity for l < 2 (stored for uniform access), solid harmonics for d
  std::vector<double> blk;
  for (int l = 0; l <= QX_LMAX_SUPPORTED + 1; ++l) s.sph_off[l] = 0;
  s.sph_off[0] = 0; blk.push_back(1.0);
  s.sph_off[1] = (int)blk.size();
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) blk.push_back(i == j ? 1.0 : 0.0);
  s.sph_off[2] = (int)blk.size();
  if (c->pure) {
    for (int k = 0; k < 30; ++k) blk.push_back(kSph2[k]);
  } else {
    for (int i = 0; i < 6; ++i)
      for (int j = 0; j < 6; ++j) blk.push_back(i == j ? 1.0 : 0.0);
  }
  s.sph_off[3] = (int)blk.size();
  s.sph = dupload(c, blk);
}

// Work matrices of qx_jk_build_noalloc: one file-scope device array per GPU
// (each device holds its own copy until the process ends), 3 Mi doubles =
// 24 MiB, enough for 5 n_cart^2 matrices up to n_cart = 792 (spherical
// bases) or 2 n_cart^2 up to n_cart = 1254 (Cartesian).  Host code never
// uses the array's name as an address: qx_initialize looks up its device
// address once per device and keeps it in g_scratch_ptr.
static __device__ __align__(256) double scratch[QX_NOALLOC_DOUBLES];

#define QX_MAX_DEVICES 64
std::mutex g_scratch_mu;
double* g_scratch_ptr[QX_MAX_DEVICES] = {};

// Device address of `scratch` on `device`, which must be current.
double* scratch_address(int device) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  QX_REQUIRE(device >= 0 && device < QX_MAX_DEVICES, QX_EINVAL, "device index beyond the scratch table");
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    QX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    QX_REQUIRE(p != nullptr, QX_EHIP, "no device address for the scratch array");
    g_scratch_ptr[device] = static_cast<double*>(p);
  }
  return g_scratch_ptr[device];
}

thread_local std::string g_init_error;

int fail(qx_ctx* c, int code, const char* msg) noexcept {
  try {
    if (c) c->err = msg; else g_init_error = msg;
  } catch (...) {
    // the message itself could not be stored; the code still reports the failure
  }
  return code;
}

int fail(qx_ctx* c, const QxError& e) noexcept { return fail(c, e.code, e.msg.c_str()); }

// Runs the body of a C-ABI entry point: every C++ exception becomes a status
// code (nothing crosses the C ABI, so nothing reaches std::terminate).
template <class F>
int guarded(qx_ctx* c, F&& body) noexcept {
  try {
    return body();
  } catch (const QxError& e) {
    return fail(c, e);
  } catch (const std::bad_alloc&) {
    return fail(c, QX_ENOMEM, "host memory allocation failed");
  } catch (const std::exception& e) {
    return fail(c, QX_EHIP, e.what());
  } catch (...) {
    return fail(c, QX_EHIP, "unexpected C++ exception");
  }
}

}  // namespace

// ============================================================== C ABI
extern "C" {

static void init_body(qx_ctx* c, int natom, const double* xyz_bohr, const double* nuclear_charges, int nshell,
                      const int* shell_l, const int* shell_atom, const int* shell_nprim, const double* exps,
                      const double* coefs, int pure, double ints_tol, int device, const int* atom_fragment);

static int init_impl(int natom, const double* xyz_bohr, const double* nuclear_charges, int nshell,
                     const int* shell_l, const int* shell_atom, const int* shell_nprim, const double* exps,
                     const double* coefs, int pure, double ints_tol, int device, const int* atom_fragment,
                     qx_ctx** out) {
  if (!out) return QX_EINVAL;
  *out = nullptr;
  qx_ctx* c = nullptr;
  const int rc = guarded(nullptr, [&]() -> int {
    try {
      c = new qx_ctx();
      for (int k = 0; k < QX_NUM_CLASSES; ++k)
        for (int pass = 0; pass < 2; ++pass) {
          c->fp32_ok[pass][k] = qx_fp32_default[k][pass];
          c->tile[pass][k] = qx_tile_default[k][pass];
          c->gwred[k] = qx_gwred_default[k];
          c->jkrows[k] = 1;
          c->gcopy[k] = qx_gcopy_default[k];
        }
      init_body(c, natom, xyz_bohr, nuclear_charges, nshell, shell_l, shell_atom, shell_nprim, exps, coefs, pure,
                ints_tol, device, atom_fragment);
    } catch (...) {
      if (c) qx_finalize(c);
      c = nullptr;
      throw;
    }
    return QX_OK;
  });
  if (rc == QX_OK) *out = c;
  return rc;
}

static void init_body(qx_ctx* c, int natom, const double* xyz_bohr, const double* nuclear_charges, int nshell,
                      const int* shell_l, const int* shell_atom, const int* shell_nprim, const double* exps,
                      const double* coefs, int pure, double ints_tol, int device, const int* atom_fragment) {
  {
    QX_REQUIRE(natom > 0 && xyz_bohr && nuclear_charges, QX_EINVAL, "natom must be positive with coordinates");
    QX_REQUIRE(nshell > 0 && shell_l && shell_atom && shell_nprim && exps && coefs, QX_EINVAL, "no shells");
    QX_REQUIRE(ints_tol > 0 && std::isfinite(ints_tol), QX_EINVAL, "ints_tol must be positive");
    // host-side tables first (a host allocation failure is reported before
    // any device work starts)
    c->natom = natom;
    c->frag.assign(natom, 0);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw QxError{QX_ENODEVICE, "no HIP device"};
    QX_REQUIRE(device >= 0 && device < ndev, QX_EINVAL, "device index out of range");
    QX_HIP(hipSetDevice(device));
    c->device = device;
    c->scratch = scratch_address(device);
    if (atom_fragment) {
      for (int a = 0; a < natom; ++a) {
        QX_REQUIRE(atom_fragment[a] >= 0, QX_EINVAL, "fragment ids must be non-negative");
        c->frag[a] = atom_fragment[a];
      }
      c->fragmented = true;
    }
    c->xyz.assign(xyz_bohr, xyz_bohr + 3 * natom);
    c->Z.assign(nuclear_charges, nuclear_charges + natom);
    for (double v : c->xyz) QX_REQUIRE(std::isfinite(v), QX_EINVAL, "non-finite coordinate");
    c->nshell = nshell;
    c->pure = pure ? 1 : 0;
    c->tol = ints_tol;
    int tp = 0, nc = 0, nb = 0;
    for (int s = 0; s < nshell; ++s) {
      QX_REQUIRE(shell_l[s] >= 0 && shell_l[s] <= QX_LMAX_SUPPORTED, QX_EUNSUPPORTED,
                 "shell angular momentum above " + std::to_string(QX_LMAX_SUPPORTED) + " is not built");
      QX_REQUIRE(shell_atom[s] >= 0 && shell_atom[s] < natom, QX_EINVAL, "shell atom index out of range");
      QX_REQUIRE(shell_nprim[s] >= 1, QX_EINVAL, "shell without primitives");
      c->l.push_back(shell_l[s]);
      c->atom.push_back(shell_atom[s]);
      c->nprim.push_back(shell_nprim[s]);
      c->poff.push_back(tp);
      c->bfc.push_back(nc);
      c->bfs.push_back(nb);
      tp += shell_nprim[s];
      nc += ncart(shell_l[s]);
      nb += nsph(shell_l[s], c->pure);
      if (shell_nprim[s] != 1) c->k1 = false;
    }
    c->ncart = nc;
    c->nbf = nb;
    c->exps.assign(exps, exps + tp);
    c->coefs.resize(tp);
    for (double v : c->exps) QX_REQUIRE(v > 0 && std::isfinite(v), QX_EINVAL, "exponents must be positive");
    for (int s = 0; s < nshell; ++s)
      normalize_shell(c->l[s], c->nprim[s], &c->exps[c->poff[s]], coefs + c->poff[s], &c->coefs[c->poff[s]]);
    static const std::vector<double> boys = boys_table();  // 0.5 ms of long double arithmetic, once per process
    c->d_boys = dupload(c, boys);
    setup_shell_tables(c);
    schwarz_and_lists(c);
    setup_jk(c);
    QX_HIP(hipDeviceSynchronize());
  }
}

int qx_initialize(int natom, const double* xyz_bohr, const double* nuclear_charges, int nshell,
                  const int* shell_l, const int* shell_atom, const int* shell_nprim, const double* exps,
                  const double* coefs, int pure, double ints_tol, int device, qx_ctx** out) {
  return init_impl(natom, xyz_bohr, nuclear_charges, nshell, shell_l, shell_atom, shell_nprim, exps, coefs, pure,
                   ints_tol, device, nullptr, out);
}

int qx_initialize_fragments(int natom, const double* xyz_bohr, const double* nuclear_charges, int nshell,
                            const int* shell_l, const int* shell_atom, const int* shell_nprim, const double* exps,
                            const double* coefs, int pure, double ints_tol, int device, const int* atom_fragment,
                            qx_ctx** out) {
  if (!atom_fragment) return QX_EINVAL;
  return init_impl(natom, xyz_bohr, nuclear_charges, nshell, shell_l, shell_atom, shell_nprim, exps, coefs, pure,
                   ints_tol, device, atom_fragment, out);
}

int qx_finalize(qx_ctx* c) {
  if (!c) return QX_EINVAL;
  (void)hipSetDevice(c->device);
  for (auto& p : c->prof_pending) {
    (void)hipEventSynchronize(p.stop);
    (void)hipEventDestroy(p.start);
    (void)hipEventDestroy(p.stop);
  }
  for (auto e : c->event_pool) (void)hipEventDestroy(e);
  (void)hipDeviceSynchronize();
  for (auto t : c->side) (void)hipStreamDestroy(t);
  for (auto e : c->fork_ev) (void)hipEventDestroy(e);
  if (c->ws_ev) (void)hipEventDestroy(c->ws_ev);
  for (int* p : {c->split.d_ck64, c->split.d_range64})
    if (p) (void)hipFree(p);
  if (c->pairm) (void)hipFree(c->pairm);
  for (void* p : c->allocs) (void)hipFree(p);
  delete c;
  return QX_OK;
}

const char* qx_last_error(const qx_ctx* c) { return c ? c->err.c_str() : g_init_error.c_str(); }

int qx_nbf(const qx_ctx* c, int* nbf, int* nc) {
  if (!c) return QX_EINVAL;
  if (nbf) *nbf = c->nbf;
  if (nc) *nc = c->ncart;
  return QX_OK;
}

int qx_schwarz_screening(qx_ctx* c, double* values, int* pairs, int* npairs) {
  if (!c) return QX_EINVAL;
  if (values) std::memcpy(values, c->Q.data(), c->Q.size() * sizeof(double));
  if (pairs) std::memcpy(pairs, c->ref_pairs.data(), c->ref_pairs.size() * sizeof(int));
  if (npairs) *npairs = (int)c->ref_pairs.size() / 2;
  return QX_OK;
}

int qx_num_quartets(const qx_ctx* c, long long* nq) {
  if (!c || !nq) return QX_EINVAL;
  *nq = c->nquart_total;
  return QX_OK;
}

long long qx_how_many_derivs(int natom, int order) {
  if (natom < 0 || order < 0) return -1;
  long long val = 1, fact = 1;
  for (int i = 0; i < order; ++i) {
    val *= 3LL * natom + i;
    fact *= i + 1;
  }
  return val / fact;
}

long long qx_generate_multi_index_lookup(int nparams, int order, int* out, long long cap) {
  if (nparams < 0 || order < 0) return -1;
  std::vector<int> cur(order, 0);
  long long count = 0;
  // combinations with replacement in lexicographic order
  if (order == 0) return 1;
  if (nparams == 0) return 0;
  while (true) {
    if (out) {
      if (count >= cap) return -1;
      for (int k = 0; k < order; ++k) out[count * order + k] = cur[k];
    }
    ++count;
    int k = order - 1;
    while (k >= 0 && cur[k] == nparams - 1) --k;
    if (k < 0) break;
    const int v = cur[k] + 1;
    for (int j = k; j < order; ++j) cur[j] = v;
  }
  return count;
}

// Workspace of one tensor pass: nslice pair matrices (or panels of one), and
// the index tables.  Up to QX_PAIRM_KEEP bytes stay with the
// context, larger ones are allocated for the call.
#define QX_PAIRM_KEEP ((size_t)1 << 30)
#define QX_PAIRM_PANEL ((size_t)64 << 20)
static const int kPairComps[6] = {1, 3, 9, 6, 18, 36};  // ss, ps, pp, ds, dp, dd

struct PairMatrix {
  QxPairIndex ix{};
  long long ld = 0, slice = 0;
  int nslice = 0;            // slices per pass
  long long panel = 0;       // M is one panel of this many rows of each slice (0: whole slices)
  double* M = nullptr;
  int* index = nullptr;
  int* fn = nullptr;
  int cleared = 0;           // M is cleared for the first pass
  bool captured = false;     // the pass is being captured
  std::unique_ptr<DevBuf> own;
};

// Device memory calls that a capture in progress, here or in another thread,
// does not refuse.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

static bool is_capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();  // the default stream while another one is captured
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

// Gives the kept workspace back; hipFree waits for passes that still read it.
static void drop_pairm(qx_ctx* c) {
  const RelaxedCapture relaxed;
  void* p = c->pairm;
  c->pairm = nullptr;
  c->pairm_bytes = 0;
  if (p) QX_HIP(hipFree(p));
}

// `bytes` of workspace, or null when the device has no room.  A captured pass
// gets its own, which stays until the context goes: replays use it whatever the
// context has done since.
static void* pairm_room(qx_ctx* c, PairMatrix& m, size_t bytes) {
  const RelaxedCapture relaxed;
  void* p = nullptr;
  if (bytes <= c->pairm_bytes && !m.captured) return c->pairm;
  if (!m.captured) drop_pairm(c);  // before the larger one, which may need its room
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (m.captured) {
    c->allocs.push_back(p);
  } else if (bytes <= QX_PAIRM_KEEP) {
    c->pairm = static_cast<double*>(p);
    c->pairm_bytes = bytes;
  } else {
    m.own.reset(new DevBuf(p));
  }
  return p;
}

// Sets m up on stream s for up to `want` slices at a time: all of them where
// the device (or pairm_limit) has room, else fewer, else row panels of as many
// slices as take 36 rows each, the components of one dd pair.
static void begin_pairm(qx_ctx* c, PairMatrix& m, int want, hipStream_t s) {
  m.captured = is_capturing(s);
  int at = 0;
  for (int X = 0; X < 6; ++X) {
    m.ix.base[X] = at;
    m.ix.cnt[X] = c->class_pair_cnt[X];
    at += kPairComps[X] * c->class_pair_cnt[X];
  }
  m.ix.base[6] = at;
  m.ld = std::max((at + 7) & ~7, 8);  // rows start on a 64-byte line
  m.slice = m.ld * m.ld;
  auto pad = [](size_t b) { return (b + 63) / 64 * 64; };
  const size_t bi = pad((size_t)c->nbf * c->nbf * sizeof(int)), bf = pad((size_t)m.ld * sizeof(int));
  const size_t tables = bi + bf;
  void* p = nullptr;
  size_t data = 0;
  for (m.nslice = want; m.nslice >= 1 && !p; m.nslice = m.nslice > 1 ? (m.nslice + 1) / 2 : 0) {
    data = (size_t)m.nslice * m.slice * sizeof(double);
    if (c->pairm_limit && data > c->pairm_limit) continue;
    if ((p = pairm_room(c, m, data + tables))) break;
  }
  const size_t row = m.ld * sizeof(double);
  if (!p) {
    // panels scatter every element to its eight places, which needs no
    // transform; a spherical tensor has always needed more room than this
    if (c->pure) throw QxError{QX_ENOMEM, "no device memory for the pair matrix of a spherical tensor"};
    for (size_t room = c->pairm_limit ? std::min(c->pairm_limit, QX_PAIRM_PANEL) : QX_PAIRM_PANEL; !p; room /= 2) {
      m.nslice = (int)std::min<size_t>(want, std::max<size_t>(1, room / (36 * row)));
      m.panel = (long long)std::max<size_t>(36, room / (m.nslice * row));
      m.slice = m.panel * m.ld;
      data = (size_t)m.nslice * m.slice * sizeof(double);
      p = pairm_room(c, m, data + tables);
      if (!p && data <= 36 * row) throw QxError{QX_ENOMEM, "no device memory for a tensor panel"};
    }
  }
  m.M = static_cast<double*>(p);
  char* q = static_cast<char*>(p) + data;
  m.index = reinterpret_cast<int*>(q);
  m.fn = reinterpret_cast<int*>(q + bi);
  if (!m.captured) order_ws(c, s);
  check_launch(qxk_pairm_tables(&c->shells, &c->pr, c->npairs, &m.ix, m.ld, m.index, m.fn, m.M, m.nslice * m.slice, &m.cleared,
                                s), "pair tables");
}

// Kets of one bra pair that a workgroup takes: enough workgroups to fill the
// device a few times over.  A K workgroup clears its K' rows, reads its density
// rows and flushes with one global atomic per element of the rows, so it takes
// QX_K_CHUNK primitive quartets or more where that leaves a quarter of
// QX_K_BLOCKS workgroups (280 functions, all K kernels of a pass: 3.35 ms with
// QX_K_BLOCKS, 2.83 ms with a quarter; of 672 functions' quartets a quarter
// would already leave CUs idle at the end: (dd|dp) 8.1 ms at half, 8.9 ms).
#define QX_K_BLOCKS 4096
#define QX_K_CHUNK 2048LL
#define QX_RYS_BLOCKS 1024LL  // quadrature workgroups below which they share primitive quartets
#define QX_SUB_LANES 65536  // lanes below which contracted quartets are shared between lanes

// Lanes that share the primitives of a contracted quartet: few quartets still
// spread over the device.
static int shared_lanes(const QxWorkHost& wh, int most) {
  return wh.prims == 1 ? 1 : (int)std::max<long long>(1, std::min<long long>({(long long)wh.prims, (long long)most, QX_SUB_LANES / wh.ncq}));
}

// The contracted list wh for a kernel of one lane per quartet in blocks of
// `block` threads, or (block = 0) of the quadrature kernels; rows: a K kernel;
// lanes: how many may share a quartet's primitives.  (Dual numbers: 81 on as
// many lanes take one round, not two: water's directional gradient 127 -> 114
// us.  The values' shorter rounds lose to the wider sums: gradient of 100 waters
// 0.11 -> 0.13 ms.)
static QxKList k_list(const qx_ctx* c, const QxWorkHost& wh, int sel, int block, bool rows, int lanes = 64) {
  QxKList kl{};
  kl.bra0 = c->class_pair_off[wh.bra_class]; kl.ket0 = c->class_pair_off[wh.ket_class];
  kl.prefix = c->d_cprefix + wh.cprefix_off;
  kl.kstart = c->fragmented ? c->d_ckstart + wh.cprefix_off : nullptr;
  kl.n64 = c->split.d_ck64 ? c->split.d_ck64 + wh.cprefix_off : nullptr;
  kl.sel = sel;
  kl.nbra = c->class_pair_cnt[wh.bra_class];
  kl.maxket = wh.maxket;
  kl.nquart = wh.ncq;
  kl.ketprim = c->class_prims[wh.ket_class];
  kl.rys = c->d_rys;
  kl.frag_atoms = c->d_frag_atoms;
  const long long prims = wh.prims;
  kl.sub = shared_lanes(wh, lanes);
  // a bra with few kets (a batch of small molecules) leaves lanes of its
  // workgroup idle: where few share so far, they do too (500 waters, minimal
  // basis: gradient 0.49 -> 0.30 ms; with more than eight the rounds saved are
  // too few: 100 waters 91 -> 97 us)
  if (block && prims > kl.sub && kl.sub <= 8)
    kl.sub = (int)std::max<long long>(kl.sub, std::min<long long>({prims, (long long)lanes, block * (long long)kl.nbra / wh.ncq}));
  const long long most = (wh.ncq + QX_K_BLOCKS - 1) / QX_K_BLOCKS;
  const long long per = std::max<long long>(rows ? std::max(most, std::min(4 * most, QX_K_CHUNK / prims)) : most, 1);
  // quadrature: in short lists as little as one step of each of a block's four
  // wavefronts (60 functions: a derivative tensor's kernels 1.27 ms in shares
  // of 32 kets, 0.70 ms so; of the long lists of 280 functions' gradient shares
  // of 40 cost 2 % more than of 64)
  static const int kPairFns[6] = {1, 3, 9, 6, 18, 36};
  const int step = 4 * (64 / kPairFns[wh.bra_class]);
  const int unit = block ? std::max(1, block / kl.sub) : per <= 16 ? std::min(step, 32) : 32;
  kl.chunk = (int)std::min<long long>((per + unit - 1) / unit * unit, 1 << 20);
  // quadrature workgroups that share a bra's primitive quartets, four or more each
  kl.psplit = 1;
  if (!block && prims >= 8) {
    const long long blocks = (long long)kl.nbra * ((kl.maxket + kl.chunk - 1) / kl.chunk);
    kl.psplit = (int)std::max<long long>(1, std::min(prims / 4, QX_RYS_BLOCKS / std::max(blocks, 1LL)));
  }
  return kl;
}

// The contracted list wh with its place in M.
static QxPairM pairm_list(const qx_ctx* c, const PairMatrix& m, const QxWorkHost& wh) {
  QxPairM pm{};
  const int X = wh.bra_class, Y = wh.ket_class;
  pm.M = m.M; pm.ld = m.ld; pm.slice = m.slice;
  pm.row0 = m.ix.base[X]; pm.rown = m.ix.cnt[X]; pm.rowp = c->class_pair_off[X];
  pm.col0 = m.ix.base[Y]; pm.coln = m.ix.cnt[Y]; pm.colp = c->class_pair_off[Y];
  pm.prefix = c->d_cprefix + wh.cprefix_off;
  pm.kstart = c->fragmented ? c->d_ckstart + wh.cprefix_off : nullptr;
  pm.nbra = c->class_pair_cnt[X];
  pm.nquart = wh.ncq;
  for (pm.sub = 1; 2 * pm.sub <= shared_lanes(wh, 64);) pm.sub *= 2;
  return pm;
}

// The same panel of a list for the quadrature kernels.
static QxKList pairm_kets(const qx_ctx* c, const QxWorkHost& wh, const QxPairM& pm) {
  QxKList kl = k_list(c, wh, 0, 0, false);
  kl.bra0 = pm.rowp;
  kl.prefix = pm.prefix;
  kl.kstart = pm.kstart;
  kl.nbra = pm.nbra;
  kl.nquart = pm.nquart;
  return kl;
}

// Evaluates the lists into nslice tensors at out: `launch(list, pm)` is one
// list's kernel; others_only: it leaves out quartets on a single atom.  Whole
// matrices are mirrored and expanded; panels are scattered.
static void run_pairm(qx_ctx* c, PairMatrix& m, int nslice, bool others_only, double* out, hipStream_t s,
                      const std::function<Launch(const QxWorkHost&, const QxPairM&)>& launch) {
  std::vector<Launch> v;
  if (m.panel == 0) {
    if (!m.cleared) check_launch(qxk_fill(m.M, nslice * m.slice, 0.0, s), "fill");
    m.cleared = 0;
    for (const auto& wh : c->work)
      if (!others_only || c->ndq_class[wh.cls] > 0) v.push_back(launch(wh, pairm_list(c, m, wh)));
    run_launches(c, v, s, "pair matrix", !m.captured);
    check_launch(qxk_pairm_ao(&c->shells, &m.ix, m.fn, m.M, m.ld, m.slice, nslice, s), "pair transform");
    check_launch(qxk_pairm_sym(c->nbf, m.M, m.ld, m.slice, nslice, &m.ix, s), "pair mirror");
    check_launch(qxk_pairm_expand(c->nbf, m.M, m.ld, m.slice, nslice, &m.ix, m.index, m.fn, out, s), "pair expand");
    return;
  }
  const size_t nc = c->ncart, n4 = nc * nc * nc * nc;
  check_launch(qxk_fill(out, (long long)(nslice * n4), 0.0, s), "fill");
  for (int X = 0; X < 6; ++X) {
    const int comps = kPairComps[X], step = (int)std::max<long long>(1, m.panel / comps);
    for (int i0 = 0; i0 < m.ix.cnt[X]; i0 += step) {
      const int cnt = std::min(step, m.ix.cnt[X] - i0);
      check_launch(qxk_fill(m.M, nslice * m.slice, 0.0, s), "fill");
      for (const auto& wh : c->work) {
        if (wh.bra_class != X) continue;
        QxPairM pm = pairm_list(c, m, wh);
        const long long* pre = c->h_cprefix.data() + wh.cprefix_off;
        pm.row0 = 0; pm.rown = cnt; pm.rowp += i0;
        pm.prefix += i0;
        if (pm.kstart) pm.kstart += i0;
        pm.nbra = cnt;
        pm.t0 = pre[i0];
        pm.nquart = pre[i0 + cnt] - pre[i0];
        v.push_back(launch(wh, pm));
      }
      run_launches(c, v, s, "pair matrix", false);
      v.clear();
      check_launch(qxk_pairm_scatter((int)nc, m.M, m.ld, m.slice, nslice, &m.ix, m.fn, X, comps, i0, cnt, out, s),
                   "pair scatter");
    }
  }
}

static void end_pairm(qx_ctx* c, PairMatrix& m, hipStream_t s) {
  if (m.captured) return;
  end_ws(c, s);
  if (m.own) QX_HIP(hipStreamSynchronize(s));  // freed on return
}

// The integral tensor (skip_single: single-atom quartets left out).
static void eri_tensor(qx_ctx* c, int skip_single, double* out, hipStream_t s) {
  PairMatrix m;
  begin_pairm(c, m, 1, s);
  QxEpiDev e{};
  e.epi = QX_EPI_PAIRM; e.nbf = c->ncart; e.natom = c->natom; e.coord = -1; e.skip_single = skip_single;
  run_pairm(c, m, 1, skip_single != 0, out, s, [&](const QxWorkHost& wh, const QxPairM& pm) {
    const QxKList kl = pairm_kets(c, wh, pm);
    return Launch{(double)pm.nquart * qx_class_table[wh.cls].eri_flops, [=](hipStream_t st) {
                    return launch_eri(c, wh.w, wh.cls, e, 0, st, c->pr, c->pp, &pm, &kl);
                  }};
  });
  end_pairm(c, m, s);
}

int qx_compute_2e_int(qx_ctx* c, double* out, void* stream) {
  if (!c || !out) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    eri_tensor(c, 0, out, (hipStream_t)stream);
    return QX_OK;
  });
}

// Adjoint-gradient kernels (every group of parts) of one quartet list; sel /
// nq: the part of the list the launch evaluates and its pseudo-pair quartet
// count.  dir: along tv instead.
static void add_grad_list(qx_ctx* c, const QxWorkHost& wh, const QxEpiDev& e, int fp32, int sel, long long nq, bool dir,
                          std::vector<Launch>& out) {
  if (wh.ncq <= 0 || nq <= 0) return;
  const QxClassEntry& ent = qx_class_table[wh.cls];
  const int block = c->tile[1][wh.cls];
  const QxKList kl = k_list(c, wh, sel, (dir ? qx_rys_h : qx_rys_g)[wh.cls] ? 0 : block, false, dir ? 128 : 64);
  const int nl = dir ? 1 : ent.ngroups;
  for (int k = 0; k < nl; ++k) {
    QxArgs a;
    a.pr = c->pr; a.pp = c->pp; a.w = wh.w; a.e = e; a.boys = c->d_boys;
    a.e.grad_wred = c->gwred[wh.cls];
    a.e.grad_copies = std::min(std::max(c->gcopy[wh.cls], 1), a.e.grad_copies);
    const int slot = QX_SLOT_DERIV(wh.cls, k, fp32 ? 1 : 0);
    auto fn = dir ? ent.hess : ent.grad[k];
    const double fl = dir ? 3.0 * ent.part_flops[0] * ent.nparts : ent.group_flops[k];
    out.push_back({(double)nq * fl, [c, a, fn, fp32, slot, nq, block, kl, dir](hipStream_t st) {
                     QxLaunch L{fp32, st, block, nullptr, &kl};
                     if (dir) return fn(&a, &L);
                     return timed_launch(c, slot, nq, st, [&] { return fn(&a, &L); });
                   }});
  }
}

// K kernel of one quartet list, as add_grad_list.
static void add_k_list(qx_ctx* c, const QxWorkHost& wh, const QxEpiDev& e, int fp32, int sel, long long nq, bool dir,
                       std::vector<Launch>& out, bool timed = true) {
  if (wh.ncq <= 0 || nq <= 0) return;
  const QxClassEntry& ent = qx_class_table[wh.cls];
  const int block = c->tile[0][wh.cls];
  const QxKList kl = k_list(c, wh, sel, (dir ? qx_rys_h : qx_rys_k)[wh.cls] ? 0 : block, true, dir ? 128 : 64);
  const int nl = dir ? 1 : ent.njk;
  for (int k = 0; k < nl; ++k) {
    QxArgs a;
    a.pr = c->pr; a.pp = c->pp; a.w = wh.w; a.e = e; a.boys = c->d_boys;
    a.e.krows = e.krows && c->jkrows[wh.cls];
    const int slot = QX_SLOT_JK(wh.cls, k, fp32 ? 1 : 0);
    auto fn = dir ? ent.jkv : ent.jk[k];
    out.push_back({(double)nq * ent.jk_flops[k], [c, a, fn, fp32, slot, nq, block, kl, dir, timed](hipStream_t st) {
                     QxLaunch L{fp32, st, block, nullptr, &kl};
                     return timed_launch(c, slot, nq, st, [&] { return fn(&a, &L); }, timed && !dir);
                   }});
  }
}

// J kernels of every bra class.  f32[X]: ket classes whose quartets beyond the
// FP32 threshold run in FP32 (mixed precision).
static void add_j_launches(qx_ctx* c, const QxEpiDev& e, const QxJList& lists, const unsigned (&f32)[6],
                           std::vector<Launch>& out, bool timed) {
  static const int order[6] = {0, 1, 2, 2, 3, 4};
  const int nu_all = lists.uoff[6];
  // a workgroup walks every ket of its bra pseudo pair; with few bras the
  // walk is shared out.  (Not further by class: every workgroup passes through
  // the code of all ket classes, and the 210 dd bras of 280 functions took
  // 587 us in 9 shares each, 160 us whole.)
  const int split = std::min(8, std::max(1, 2048 / std::max(nu_all, 1)));
  const int block = nu_all / split >= 512 ? 256 : 64;
  for (int X = 5; X >= 0; --X) {
    const long long nu = lists.uoff[X + 1] - lists.uoff[X];
    if (nu <= 0) continue;
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1 && f32[X] == 0) continue;
      const int type = e.tv ? 2 : pass;
      QxArgs a;
      a.pr = c->pr; a.pp = c->pp; a.w = QxWorkDev{}; a.e = e; a.boys = c->d_boys;
      QxJList jl = lists;
      jl.X = X;
      jl.f32_classes = f32[X];
      jl.n64 = c->split.d_range64;
      auto fn = qx_j_table[order[X]];
      const int slot = QX_SLOT_JK(class_index(X, X), 1, pass);
      const double flops = 100.0 + 25.0 * (order[X] + 1) * (order[X] + 2);
      out.push_back({(double)nu * nu_all * flops, [c, a, jl, fn, type, block, split, slot, nu, nu_all, timed](hipStream_t st) {
                       return timed_launch(c, slot, nu * nu_all, st, [&] { return fn(&a, &jl, type, block, split, st); },
                                           timed && type != 2);
                     }});
    }
  }
}

// Mixed precision, per quartet list i of the split (pass 0 J/K, 1
// gradient): 0 = FP64 kernels, 1 = FP32 kernels, 2 = two launches masked to
// the FP64 and FP32 kets.  FP32 is used in the classes whose policy admits it
// and only when at least QX_MIXED_MIN_FRAC of the list's primitive quartets
// are below the threshold: a masked launch pair runs every wave that holds
// quartets of both kinds twice, which a small FP32 share does not repay.
#define QX_MIXED_MIN_FRAC 0.25
static int mixed_mode(const qx_ctx* c, size_t i, int pass) {
  const auto& S = c->split;
  const long long p64 = S.pq64[i], p32 = S.pq32[i];
  if (pass == 1 && qx_rys_g[c->work[i].cls]) return 0;  // the quadrature gradient has no FP32 form
  if (!c->fp32_ok[pass][c->work[i].cls] || p32 < QX_MIXED_MIN_FRAC * (double)(p64 + p32)) return 0;
  return p64 == 0 ? 1 : 2;
}

static void add_mixed_launches(qx_ctx* c, double thr, int pass, const QxEpiDev& e, std::vector<Launch>& out) {
  build_split(c, thr);
  const auto& S = c->split;
  auto add = [&](const QxWorkHost& wh, int f32, int sel, long long nq) {
    if (pass == 0) add_k_list(c, wh, e, f32, sel, nq, false, out);
    else add_grad_list(c, wh, e, f32, sel, nq, false, out);
  };
  for (size_t i = 0; i < c->work.size(); ++i) {
    const QxWorkHost& wh = c->work[i];
    switch (mixed_mode(c, i, pass)) {
      case 0: add(wh, 0, 0, wh.w.nquart); break;
      case 1: add(wh, 1, 0, wh.w.nquart); break;
      default:
        add(wh, 0, 1, S.pq64[i]);
        add(wh, 1, 2, S.pq32[i]);
    }
  }
}

// One list's derivative kernel (fp32 = 2: along e.tv) into the pair matrix.
static Launch deri_launch(qx_ctx* c, const QxWorkHost& wh, const QxPairM& pm, const QxEpiDev& e, int type) {
  const QxKList kl = pairm_kets(c, wh, pm);
  QxArgs a;
  a.pr = c->pr; a.pp = c->pp; a.w = wh.w; a.e = e; a.boys = c->d_boys;
  const QxClassEntry& ent = qx_class_table[wh.cls];
  return Launch{(double)pm.nquart * ent.part_flops[0] * ent.nparts, [=](hipStream_t st) {
                  QxLaunch L{type, st, 0, &pm, &kl};
                  return qx_class_table[wh.cls].deri(&a, &L);
                }};
}

// First-derivative tensor slices: all 3N (coord < 0) or one, as many at a
// time as begin_pairm found room for.
static void deriv_tensor(qx_ctx* c, int coord, double* out, hipStream_t s) {
  const int nslices = coord >= 0 ? 1 : 3 * c->natom;
  const size_t nb = c->nbf, nb4 = nb * nb * nb * nb;
  PairMatrix m;
  begin_pairm(c, m, nslices, s);
  const int group = m.nslice;
  for (int y0 = 0; y0 < nslices; y0 += group) {
    const int ny = std::min(group, nslices - y0);
    QxEpiDev e{};
    e.epi = QX_EPI_PAIRM; e.nbf = c->ncart; e.natom = c->natom; e.coord = coord;
    if (ny < nslices) {
      e.slice0 = y0;
      e.nslice = ny;
    }
    run_pairm(c, m, ny, true, out + (size_t)y0 * nb4, s, [&](const QxWorkHost& wh, const QxPairM& pm) {
      return deri_launch(c, wh, pm, e, 0);
    });
  }
  end_pairm(c, m, s);
}

// Index of the coordinate pair (x <= y) among the m(m+1)/2 pairs in
// generate_multi_index_lookup(m, 2) order.
static long long pair_index(int x, int y, int m) {
  return (long long)x * m - (long long)x * (x - 1) / 2 + (y - x);
}

// Second-derivative tensor: for each nuclear coordinate x the derivative
// kernels in dual numbers along e_x give d2(ab|cd)/dx dy for every y; slices
// y >= x are the consecutive pairs (x, y) (all pairs when want < 0, else only
// pair `want` into slice 0), as many at a time as there is room for.  Quartets
// on one atom are skipped, like the first-derivative tensor.
static void deriv2_tensor(qx_ctx* c, long long want, double* out, hipStream_t s) {
  const size_t nb = c->nbf, nb4 = nb * nb * nb * nb;
  const int m = 3 * c->natom;
  PairMatrix pmx;
  begin_pairm(c, pmx, want >= 0 ? 1 : m, s);
  const int room = pmx.nslice;
  struct Pass {
    int x, y0, ny;
  };
  std::vector<Pass> passes;
  for (int x = 0; x < m; ++x)
    for (int y = x; y < m;) {
      if (want >= 0) {
        if (pair_index(x, y, m) == want) passes.push_back({x, y, 1});
        ++y;
        continue;
      }
      const int ny = std::min(room, m - y);
      passes.push_back({x, y, ny});
      y += ny;
    }
  std::vector<double> tv((size_t)m * m, 0.0);
  for (int x = 0; x < m; ++x) tv[(size_t)x * m + x] = 1.0;
  DevBuf dtv(tv.size() * sizeof(double));
  QX_HIP(hipMemcpy(dtv.d(), tv.data(), tv.size() * sizeof(double), hipMemcpyHostToDevice));
  for (const Pass& ps : passes) {
    QxEpiDev e{};
    e.epi = QX_EPI_PAIRM; e.nbf = c->ncart; e.natom = c->natom; e.coord = -1;
    e.tv = dtv.d() + (size_t)ps.x * m;
    e.slice0 = ps.y0;
    e.nslice = ps.ny;
    double* dst = out + (want >= 0 ? 0 : (size_t)pair_index(ps.x, ps.y0, m) * nb4);
    run_pairm(c, pmx, ps.ny, true, dst, s, [&](const QxWorkHost& wh, const QxPairM& pm) {
      return deri_launch(c, wh, pm, e, 2);
    });
  }
  end_pairm(c, pmx, s);
  QX_HIP(hipStreamSynchronize(s));  // dtv is freed on return
}

int qx_eri_deriv_core(qx_ctx* c, int order, double* out, void* stream) {
  if (!c || !out) return QX_EINVAL;
  if (order != 1 && order != 2) {
    return fail(c, QX_EUNSUPPORTED, "eri_deriv_core: deriv_order 1 and 2 are built");
  }
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    if (order == 1) deriv_tensor(c, -1, out, (hipStream_t)stream);
    else deriv2_tensor(c, -1, out, (hipStream_t)stream);
    return QX_OK;
  });
}

int qx_compute_2e_deriv(qx_ctx* c, const int* dv, int len, double* out, void* stream) {
  if (!c || !out || !dv) return QX_EINVAL;
  if (len != 3 * c->natom) {
    return fail(c, QX_EINVAL, "compute_2e_deriv: deriv_vec length must be 3*natom");
  }
  int order = 0, coord = -1, c2[2] = {-1, -1}, k = 0;
  for (int i = 0; i < len; ++i) {
    if (dv[i] < 0) return fail(c, QX_EINVAL, "compute_2e_deriv: negative deriv_vec entry");
    order += dv[i];
    if (dv[i]) coord = i;
    for (int r = 0; r < dv[i] && k < 2; ++r) c2[k++] = i;
  }
  if (order > 2) {
    return fail(c, QX_EUNSUPPORTED, "compute_2e_deriv: deriv_vec orders 0, 1 and 2 are built");
  }
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    if (order == 0) {
      // the reference's order-0 call returns buffer 0 of a deriv-0 engine, i.e.
      // the integrals, with single-atom quartets skipped (libint_interface.cc:1180-1185)
      eri_tensor(c, 1, out, s);
      return QX_OK;
    }
    if (order == 1) deriv_tensor(c, coord, out, s);
    else deriv2_tensor(c, pair_index(c2[0], c2[1], len), out, s);
    return QX_OK;
  });
}

// Whether the caller left the per-class tuning of the s and p classes' kernels
// (pass 0 J/K, 1 gradient) as it is built in: one launch for all has none.
static bool default_tuning(const qx_ctx* c, int pass) {
  for (int k = 0; k < 6; ++k) {
    if (c->tile[pass][k] != qx_tile_default[k][pass]) return false;
    if (pass == 0 && !c->jkrows[k]) return false;
    if (pass == 1 && (c->gwred[k] != qx_gwred_default[k] || c->gcopy[k] != qx_gcopy_default[k])) return false;
  }
  return true;
}

// The lists of a pass as one launch, where no shell is above p and the whole
// pass has at most QX_SMALL_QUARTETS primitive quartets: minimal basis, 3 atoms
// 49 us against 128 in separate launches, 8 atoms (0.7 million) 92 against 135,
// 12 atoms (3.4 million) 206 against 201, 16 atoms 482 against 415, where the
// registers of the largest class and one block size for all cost more than the
// launches.
#define QX_SMALL_QUARTETS 2000000
static bool small_pass(qx_ctx* c, const QxEpiDev& e, const QxJList& jl, bool timed, QxSmall& sm, size_t& lds) {
  if ((timed && c->profiling) || !e.krows || !default_tuning(c, 0) || c->class_pair_cnt[3] + c->class_pair_cnt[4] + c->class_pair_cnt[5] > 0) return false;
  if (c->npq_total > QX_SMALL_QUARTETS) return false;
  sm = QxSmall{};
  long long blocks[9] = {};
  lds = 0;
  const size_t W = e.kcols > 0 ? e.kcols : e.nbf;
  for (const auto& wh : c->work) {
    const int at = wh.cls;  // s and p classes: 0000, 1000, 1010, 1100, 1110, 1111
    const QxKList kl = k_list(c, wh, 0, QX_SMALL_BLOCK, true);
    sm.k[at] = kl;
    if (kl.nquart > 0 && kl.maxket > 0) blocks[at] = (long long)kl.nbra * ((kl.maxket + kl.chunk - 1) / kl.chunk);
    lds = std::max(lds, 2 * (ncart(at < 1 ? 0 : 1) + ncart(at < 3 ? 0 : 1)) * W * sizeof(double));
  }
  if (lds > QX_K_STAGE_MAX) return false;
  sm.split = std::min(8, std::max(1, 2048 / std::max(jl.uoff[6], 1)));
  for (int X = 0; X < 3; ++X) {
    sm.j[X] = jl;
    sm.j[X].X = X;
    blocks[6 + X] = (long long)(jl.uoff[X + 1] - jl.uoff[X]) * sm.split;
  }
  long long end = 0;
  for (int i = 0; i < 9; ++i) {
    end += blocks[i];
    if (end > 0x7fffffff) return false;
    sm.end[i] = (int)end;
  }
  return true;
}

// The same for the gradient: minimal basis, 3 atoms 44 us against 114 in
// separate launches, 8 atoms 99 against 127, 16 atoms (10 million primitive
// quartets) 366 against 402, 20 atoms 734 against 672.
#define QX_SMALL_GRAD_QUARTETS 10000000
static_assert(QX_SMALL_GRADS <= 16, "lists of the one-launch gradient");
static bool small_grad(const qx_ctx* c, QxSmallGrad& sm) {
  if (c->profiling || !default_tuning(c, 1) || c->class_pair_cnt[3] + c->class_pair_cnt[4] + c->class_pair_cnt[5] > 0)
    return false;
  if (c->npq_total > QX_SMALL_GRAD_QUARTETS) return false;
  sm = QxSmallGrad{};
  long long blocks[6] = {}, end = 0;
  for (const auto& wh : c->work) {
    const QxKList kl = k_list(c, wh, 0, QX_SMALL_BLOCK, false);
    sm.k[wh.cls] = kl;
    if (kl.nquart > 0 && kl.maxket > 0) blocks[wh.cls] = (long long)kl.nbra * ((kl.maxket + kl.chunk - 1) / kl.chunk);
  }
  for (int i = 0; i < QX_SMALL_GRADS; ++i) {
    end += blocks[qx_small_grad_class[i]];
    if (end > 0x7fffffff) return false;
    sm.end[i] = (int)end;
  }
  return true;
}

// J and K of D with work matrices w (2 n_cart^2 doubles, 3 for a spherical
// basis), or (tv) of the integrals' derivative along tv.  herm: Hermite
// densities and potentials (2 nherm doubles) of a pass that may run beside the
// context's other passes: it touches no memory of theirs, keeps to stream s and
// uses no events.  Null: the context's, spread over the side streams.
static void jk_pass(qx_ctx* c, double* w, const double* D, double* J, double* K, int precision, double thr,
                    const int* frag_skip, const double* tv, hipStream_t s, double* herm = nullptr) {
  const size_t nc = c->ncart, n2 = nc * nc;
  double *Jc = w, *Kp = w + n2;
  QxArgs a;
  a.pr = c->pr; a.pp = c->pp; a.w = QxWorkDev{}; a.boys = c->d_boys;
  QxEpiDev& e = a.e;
  e = QxEpiDev{};
  e.epi = QX_EPI_JK; e.nbf = (int)nc; e.natom = c->natom; e.coord = -1; e.D = D; e.J = Jc; e.K = Kp;
  if (c->pure) {
    check_launch(qxk_ao_to_cart_mat(&c->shells, D, w + 2 * n2, s), "ao_to_cart");
    e.D = w + 2 * n2;
  }
  set_krows(c, e);
  if (frag_skip) {
    e.frag_skip = frag_skip;
    e.pair_frag = c->d_pair_frag;
  }
  e.tv = tv;
  QxJList jl = c->jlist;
  const bool alone = herm != nullptr;
  if (alone) {
    jl.H = herm;
    jl.P = herm + c->nherm;
    jl.Hd = jl.Pd = nullptr;
  }
  check_launch(qxk_jk_begin(&a, &jl, c->nherm, Jc, Kp, (long long)n2, s), "jk_begin");
  std::vector<Launch> v;
  unsigned f32[6] = {};
  QxSmall sm;
  size_t lds = 0;
  if (precision == QX_PREC_FP64 && !tv && small_pass(c, e, jl, !alone, sm, lds)) {
    check_launch(qx_launch_small(&a, &sm, (unsigned)lds, s), "jk_build");
    check_launch(qxk_j_finish(&a, &jl, Jc, s), "j_finish");
    check_launch(qxk_jk_finish(&c->shells, Jc, Kp, J, K, s), "jk_finish");
    return;
  }
  if (precision == QX_PREC_MIXED) {
    add_mixed_launches(c, thr, 0, e, v);
    for (size_t i = 0; i < c->work.size(); ++i)
      if (mixed_mode(c, i, 0) != 0) {
        const QxWorkHost& wh = c->work[i];
        f32[wh.bra_class] |= 1u << wh.ket_class;
        f32[wh.ket_class] |= 1u << wh.bra_class;
      }
  } else {
    for (const auto& wh : c->work) add_k_list(c, wh, e, 0, 0, wh.w.nquart, tv != nullptr, v, !alone);
  }
  add_j_launches(c, e, jl, f32, v, !alone);
  run_launches(c, v, s, "jk_build", !alone);
  check_launch(qxk_j_finish(&a, &jl, Jc, s), "j_finish");
  check_launch(qxk_jk_finish(&c->shells, Jc, Kp, J, K, s), "jk_finish");
}

int qx_jk_build(qx_ctx* c, const double* D, double* J, double* K, int precision, double thr, void* stream) {
  return qx_jk_build_masked(c, D, J, K, precision, thr, nullptr, stream);
}

int qx_jk_build_masked(qx_ctx* c, const double* D, double* J, double* K, int precision, double thr,
                       const int* frag_skip, void* stream) {
  if (!c || !D || !J || !K) return QX_EINVAL;
  if (frag_skip && !c->fragmented) return QX_EINVAL;
  if (precision != QX_PREC_FP64 && precision != QX_PREC_MIXED) return QX_EINVAL;
  if (precision == QX_PREC_MIXED && !(thr >= 0.0 && std::isfinite(thr))) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    double* w = begin_ws(c, s);
    jk_pass(c, w, D, J, K, precision, thr, frag_skip, nullptr, s);
    end_ws(c, s);
    return QX_OK;
  });
}

// qx_jk_build (FP64) without any device allocation: the J'/K' work
// matrices live in the scratch array, the Hermite densities and potentials in
// memory of the context that only this call writes, every kernel runs in turn
// on the caller's stream (no side streams, events or timing), and the pass's
// first kernel clears what it accumulates into.  So it may overlap the
// context's other passes; two of these calls that overlap on one GPU share the
// array and race.
int qx_jk_build_noalloc(qx_ctx* c, const double* D, double* J, double* K, void* stream) {
  if (!c || !D || !J || !K) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    const size_t need = noalloc_doubles(c);
    if (need > QX_NOALLOC_DOUBLES)
      throw QxError{QX_EINVAL, "jk_build_noalloc: " + std::to_string(need) + " doubles of work matrices (" +
                                   std::to_string(c->ncart) + " Cartesian functions) exceed the " +
                                   std::to_string(QX_NOALLOC_DOUBLES) + "-double scratch array"};
    QX_REQUIRE(c->scratch != nullptr, QX_EHIP, "jk_build_noalloc: scratch array not set up");
    jk_pass(c, c->scratch, D, J, K, QX_PREC_FP64, 0.0, nullptr, nullptr, s, c->d_herm_own);
    return QX_OK;
  });
}

long long qx_jk_noalloc_capacity(void) { return (long long)QX_NOALLOC_DOUBLES; }

int qx_eri_grad(qx_ctx* c, const double* D, double* grad, int precision, double thr, void* stream) {
  if (!c || !D || !grad) return QX_EINVAL;
  if (precision != QX_PREC_FP64 && precision != QX_PREC_MIXED) return QX_EINVAL;
  if (precision == QX_PREC_MIXED && !(thr >= 0.0 && std::isfinite(thr))) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    const size_t nc = c->ncart, n2 = nc * nc;
    double* w = begin_ws(c, s);
    const double* Dcart = D;
    if (c->pure) {
      check_launch(qxk_ao_to_cart_mat(&c->shells, D, w + 2 * n2, s), "ao_to_cart");
      Dcart = w + 2 * n2;
    }
    QxEpiDev e{};
    e.epi = QX_EPI_GRAD; e.nbf = (int)nc; e.natom = c->natom; e.coord = -1; e.D = Dcart;
    e.grad = begin_grad_copies(c, s);
    e.grad_copies = QX_GRAD_COPIES;
    e.grad_win = c->grad_win;
    e.pair_frag = c->d_pair_frag;
    QxSmallGrad sm;
    if (precision == QX_PREC_FP64 && small_grad(c, sm)) {
      QxArgs a;
      a.pr = c->pr; a.pp = c->pp; a.w = QxWorkDev{}; a.e = e; a.boys = c->d_boys;
      a.e.grad_wred = 1;
      check_launch(qx_launch_small_grad(&a, &sm, s), "eri_grad");
      check_launch(qxk_add_copies(c->gcopies, QX_GRAD_COPIES, 3 * c->natom, grad, s), "gradient copies");
      end_ws(c, s);
      return QX_OK;
    }
    std::vector<Launch> v;
    if (precision == QX_PREC_MIXED) {
      add_mixed_launches(c, thr, 1, e, v);
    } else {
      for (const auto& wh : c->work) add_grad_list(c, wh, e, 0, 0, wh.w.nquart, false, v);
    }
    run_launches(c, v, s, "eri_grad", true);
    check_launch(qxk_add_copies(c->gcopies, QX_GRAD_COPIES, 3 * c->natom, grad, s), "gradient copies");
    end_ws(c, s);
    return QX_OK;
  });
}

// Forward-over-reverse piece of the Hessian-vector product: the adjoint
// contraction of the second-derivative integrals along v,
// out[y] += sum_pqrs Gamma(D)_pqrs d/dv d(pq|rs)/dR_y, Gamma = 2 D_pq D_rs -
// D_pr D_qs (the gradient kernels in dual numbers, nothing stored).
int qx_eri_hess_dir(qx_ctx* c, const double* D, const double* v, double* out, void* stream) {
  if (!c || !D || !v || !out) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    const size_t nc = c->ncart, n2 = nc * nc;
    double* w = begin_ws(c, s);
    const double* Dcart = D;
    if (c->pure) {
      check_launch(qxk_ao_to_cart_mat(&c->shells, D, w + 2 * n2, s), "ao_to_cart");
      Dcart = w + 2 * n2;
    }
    QxEpiDev e{};
    e.epi = QX_EPI_GRAD; e.nbf = (int)nc; e.natom = c->natom; e.coord = -1; e.D = Dcart; e.tv = v;
    e.grad = begin_grad_copies(c, s);
    e.grad_copies = QX_GRAD_COPIES;
    e.grad_win = c->grad_win;
    e.pair_frag = c->d_pair_frag;
    std::vector<Launch> L;
    for (const auto& wh : c->work) add_grad_list(c, wh, e, 0, 0, wh.w.nquart, true, L);
    run_launches(c, L, s, "eri_hess_dir", true);
    check_launch(qxk_add_copies(c->gcopies, QX_GRAD_COPIES, 3 * c->natom, out, s), "gradient copies");
    end_ws(c, s);
    return QX_OK;
  });
}

// J and K of the directional derivative of the integrals along v at fixed D:
// J_pq = sum_rs (d/dv (pq|rs)) D_rs, K_pq = sum_rs (d/dv (pr|qs)) D_rs (the
// derivative Fock matrix of the coupled-perturbed equations).
int qx_jk_deriv_dir(qx_ctx* c, const double* D, const double* v, double* J, double* K, void* stream) {
  if (!c || !D || !v || !J || !K) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    double* w = begin_ws(c, s);
    jk_pass(c, w, D, J, K, QX_PREC_FP64, 0.0, nullptr, v, s);
    end_ws(c, s);
    return QX_OK;
  });
}

// Every shell-pair class of a one-electron pass.
static void run_oei(qx_ctx* c, QxOei& a, int mode, hipStream_t s, const char* what) {
  a.sh = c->shells;
  a.boys = c->d_boys;
  for (int la = 0, X = 0; la <= QX_LMAX_SUPPORTED; ++la)
    for (int lb = 0; lb <= la; ++lb, ++X) {
      a.la = c->d_shell_by_l + c->l_off[la]; a.nla = c->l_off[la + 1] - c->l_off[la];
      a.lb = c->d_shell_by_l + c->l_off[lb]; a.nlb = c->l_off[lb + 1] - c->l_off[lb];
      const long long np = la == lb ? (long long)a.nla * (a.nla + 1) / 2 : (long long)a.nla * a.nlb;
      QX_REQUIRE(np <= 0x7fffffff, QX_EUNSUPPORTED, "too many shell pairs for a one-electron pass");
      a.npair = (int)np;
      check_launch(qx_oei_table[X](&a, mode, s), what);
    }
}

int qx_oei(qx_ctx* c, double* S, double* T, double* V, void* stream) {
  if (!c || !S || !T || !V) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    const size_t n2 = (size_t)c->ncart * c->ncart;
    QxOei a{};
    a.S = S; a.T = T; a.V = V;
    if (!c->pure) {
      run_oei(c, a, 0, s, "oei");
    } else {
      double* w = begin_ws(c, s);
      a.S = w; a.T = w + n2; a.V = w + 2 * n2;
      run_oei(c, a, 0, s, "oei");
      double* const out[3] = {S, T, V};
      check_launch(qxk_cart_to_ao_mats(&c->shells, w, n2, out, 3, s), "cart_to_ao");
      end_ws(c, s);
    }
    return QX_OK;
  });
}

// grad += Pd . d(T+V)/dR + Wd . dS/dR, or (v) its derivative along v.
static void oei_contract(qx_ctx* c, const double* Pd, const double* Wd, const double* v, double* grad, hipStream_t s,
                         const char* what) {
  const size_t n2 = (size_t)c->ncart * c->ncart;
  QxOei a{};
  a.Pd = Pd; a.Wd = Wd; a.grad = grad; a.tv = v;
  if (c->pure) {
    double* w = begin_ws(c, s);
    const double* const in[2] = {Pd, Wd};
    check_launch(qxk_ao_to_cart_mats(&c->shells, in, w, n2, 2, s), "ao_to_cart");
    a.Pd = w; a.Wd = w + n2;
  }
  run_oei(c, a, v ? 2 : 1, s, what);
  if (c->pure) end_ws(c, s);
}

int qx_oei_grad(qx_ctx* c, const double* Pd, const double* Wd, double* grad, void* stream) {
  if (!c || !Pd || !Wd || !grad) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    oei_contract(c, Pd, Wd, nullptr, grad, s, "oei_grad");
    return QX_OK;
  });
}

// One-electron piece of the Hessian-vector product: grad[3N] +=
// sum_pq Pd_pq d/dv d(T+V)_pq/dR + Wd_pq d/dv dS_pq/dR (tangent mode of the
// one-electron gradient kernel; v: 3N device vector).
int qx_oei_hess_dir(qx_ctx* c, const double* Pd, const double* Wd, const double* v, double* grad, void* stream) {
  if (!c || !Pd || !Wd || !v || !grad) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    oei_contract(c, Pd, Wd, v, grad, s, "oei_hess_dir");
    return QX_OK;
  });
}

int qx_oei_deriv(qx_ctx* c, double* dS, double* dT, double* dV, void* stream) {
  if (!c || !dS || !dT || !dV) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    const long long m = 3LL * c->natom, nc2 = (long long)c->ncart * c->ncart, nb2 = (long long)c->nbf * c->nbf;
    std::unique_ptr<DevBuf> tmp(c->pure ? new DevBuf((size_t)(3 * m * nc2) * sizeof(double)) : nullptr);
    double* cS = c->pure ? tmp->d() : dS;
    double* cT = c->pure ? tmp->d() + m * nc2 : dT;
    double* cV = c->pure ? tmp->d() + 2 * m * nc2 : dV;
    check_launch(qxk_fill(cS, m * nc2, 0.0, s), "fill");
    check_launch(qxk_fill(cT, m * nc2, 0.0, s), "fill");
    check_launch(qxk_fill(cV, m * nc2, 0.0, s), "fill");
    check_launch(qxk_oei_deriv(&c->shells, cS, cT, cV, s), "oei_deriv");
    if (c->pure) {
      // every coordinate slice Cartesian -> AO
      for (long long x = 0; x < m; ++x) {
        check_launch(qxk_cart_to_ao_mat(&c->shells, cS + x * nc2, dS + x * nb2, s), "cart_to_ao");
        check_launch(qxk_cart_to_ao_mat(&c->shells, cT + x * nc2, dT + x * nb2, s), "cart_to_ao");
        check_launch(qxk_cart_to_ao_mat(&c->shells, cV + x * nc2, dV + x * nb2, s), "cart_to_ao");
      }
      QX_HIP(hipStreamSynchronize(s));
    }
    return QX_OK;
  });
}

int qx_store_size(const qx_ctx* c, long long* nd) {
  if (!c || !nd) return QX_EINVAL;
  *nd = c->store_total;
  return QX_OK;
}

int qx_eri_store(qx_ctx* c, double* out, void* stream) {
  if (!c || !out) return QX_EINVAL;
  if (!c->k1) {
    return fail(c, QX_EUNSUPPORTED, "eri_store: single-primitive shells only");
  }
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    hipStream_t s = (hipStream_t)stream;
    QxEpiDev e{};
    e.epi = QX_EPI_STORE; e.nbf = c->ncart; e.natom = c->natom; e.coord = -1; e.out = out;
    for (auto& wh : c->work) {
      const QxKList kl = k_list(c, wh, 0, 0, false);
      check_launch(launch_eri(c, wh.w, wh.cls, e, 0, s, c->pr, c->pp, nullptr, &kl), "eri_store");
    }
    return QX_OK;
  });
}

int qx_store_lists(const qx_ctx* c, int* nlists, int* l4, long long* base, long long* nquart) {
  if (!c || !nlists) return QX_EINVAL;
  *nlists = (int)c->work.size();
  for (size_t k = 0; k < c->work.size(); ++k) {
    const QxWorkHost& wh = c->work[k];
    const QxClassEntry& e = qx_class_table[wh.cls];
    if (l4) {
      l4[4 * k] = e.la; l4[4 * k + 1] = e.lb; l4[4 * k + 2] = e.lc; l4[4 * k + 3] = e.ld;
    }
    if (base) base[k] = wh.w.store_base;
    if (nquart) nquart[k] = wh.w.nquart;
  }
  return QX_OK;
}

int qx_store_quartet_pairs(const qx_ctx* c, int list, int* p1, int* p2) {
  if (!c || !p1 || !p2 || list < 0 || list >= (int)c->work.size()) return QX_EINVAL;
  const QxWorkHost& wh = c->work[list];
  const long long* pre = c->h_prefix.data() + wh.prefix_off;
  const int* kst = c->h_kstart.data() + c->h_kstart_off[list];
  for (int lo = 0; lo < wh.w.nbra; ++lo) {
    const int u1 = wh.w.bra_off + lo;
    for (long long t = pre[lo]; t < pre[lo + 1]; ++t) {
      const int u2 = wh.w.ket_off + kst[lo] + (int)(t - pre[lo]);
      p1[t] = c->h_ppair[u1];
      p2[t] = c->h_ppair[u2];
    }
  }
  return QX_OK;
}

int qx_pair_shells(const qx_ctx* c, int* npairs, int* sa, int* sb) {
  if (!c || !npairs) return QX_EINVAL;
  *npairs = c->npairs;
  for (int i = 0; i < c->npairs; ++i) {
    if (sa) sa[i] = c->h_pair_sa[i];
    if (sb) sb[i] = c->h_pair_sb[i];
  }
  return QX_OK;
}

int qx_num_classes(void) { return QX_NUM_CLASSES; }

int qx_profile_slots(void) { return QX_PROFILE_SLOTS; }

int qx_profile_slot(int slot, int* kind, int* cls, int* part, int* fp32) {
  if (slot < 0 || slot >= QX_PROFILE_SLOTS) return QX_EINVAL;
  int k, c, p = 0, f;
  if (slot < 2 * QX_NUM_CLASSES_MAX) {
    k = 0; f = slot / QX_NUM_CLASSES_MAX; c = slot % QX_NUM_CLASSES_MAX;
  } else if (slot < QX_SLOT_JK0) {
    const int r = slot - 2 * QX_NUM_CLASSES_MAX;
    k = 1; p = r % QX_DPARTS_CAP;
    const int fc = r / QX_DPARTS_CAP;
    f = fc / QX_NUM_CLASSES_MAX; c = fc % QX_NUM_CLASSES_MAX;
  } else {
    const int r = slot - QX_SLOT_JK0;
    k = 2; p = r % QX_JKPARTS_CAP;
    const int fc = r / QX_JKPARTS_CAP;
    f = fc / QX_NUM_CLASSES_MAX; c = fc % QX_NUM_CLASSES_MAX;
  }
  if (kind) *kind = k;
  if (cls) *cls = c;
  if (part) *part = p;
  if (fp32) *fp32 = f;
  return QX_OK;
}

int qx_mixed_quartets(qx_ctx* c, double thr, long long* n64, long long* n32) {
  return qx_mixed_pass_quartets(c, thr, -1, n64, n32);
}

int qx_mixed_pass_quartets(qx_ctx* c, double thr, int pass, long long* n64, long long* n32) {
  if (!c || !(thr >= 0.0 && std::isfinite(thr)) || pass < -1 || pass > 1) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    build_split(c, thr);
    const auto& S = c->split;
    long long a = 0, b = 0;
    for (size_t i = 0; i < c->work.size(); ++i) {
      const bool f32 = pass < 0 || mixed_mode(c, i, pass) != 0;
      a += f32 ? S.cq64[i] : S.cq64[i] + S.cq32[i];
      b += f32 ? S.cq32[i] : 0;
    }
    if (n64) *n64 = a;
    if (n32) *n32 = b;
    return QX_OK;
  });
}

int qx_set_class_tiles(qx_ctx* c, int pass, const int* block) {
  if (!c || pass < 0 || pass > 1) return QX_EINVAL;
  if (block)
    for (int k = 0; k < QX_NUM_CLASSES; ++k)
      if (block[k] < 64 || block[k] > QX_BLOCK_MAX || block[k] % 64) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) c->tile[pass][k] = block ? block[k] : qx_tile_default[k][pass];
  return QX_OK;
}

int qx_set_grad_wave_reduce(qx_ctx* c, const int* flags) {
  if (!c) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) c->gwred[k] = flags ? (flags[k] != 0) : qx_gwred_default[k];
  return QX_OK;
}

int qx_set_grad_copies(qx_ctx* c, const int* copies) {
  if (!c) return QX_EINVAL;
  if (copies)
    for (int k = 0; k < QX_NUM_CLASSES; ++k)
      if (copies[k] < 1 || copies[k] > QX_GRAD_COPIES) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) c->gcopy[k] = copies ? copies[k] : qx_gcopy_default[k];
  return QX_OK;
}

int qx_set_jk_rows(qx_ctx* c, const int* flags) {
  if (!c) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) c->jkrows[k] = flags ? (flags[k] != 0) : 1;
  return QX_OK;
}

int qx_get_jk_rows(const qx_ctx* c, int* flags) {
  if (!c || !flags) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) flags[k] = c->jkrows[k];
  return QX_OK;
}

int qx_set_grad_window(qx_ctx* c, int atoms) {
  if (!c || atoms < 0 || 3 * atoms > QX_GRAD_LDS) return QX_EINVAL;
  c->grad_win = 3 * atoms;
  return QX_OK;
}

int qx_get_grad_window(const qx_ctx* c, int* atoms) {
  if (!c || !atoms) return QX_EINVAL;
  *atoms = (c->grad_win > 0 ? c->grad_win : QX_GRAD_LDS) / 3;
  return QX_OK;
}

int qx_get_grad_copies(const qx_ctx* c, int* copies) {
  if (!c || !copies) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) copies[k] = c->gcopy[k];
  return QX_OK;
}

int qx_get_grad_wave_reduce(const qx_ctx* c, int* flags) {
  if (!c || !flags) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) flags[k] = c->gwred[k];
  return QX_OK;
}

int qx_get_class_tiles(const qx_ctx* c, int pass, int* block) {
  if (!c || !block || pass < 0 || pass > 1) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) block[k] = c->tile[pass][k];
  return QX_OK;
}

int qx_set_fp32_classes(qx_ctx* c, int pass, const int* flags) {
  if (!c || pass < 0 || pass > 1) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) c->fp32_ok[pass][k] = flags ? (flags[k] != 0) : qx_fp32_default[k][pass];
  return QX_OK;
}

int qx_get_fp32_classes(const qx_ctx* c, int pass, int* flags) {
  if (!c || !flags || pass < 0 || pass > 1) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) flags[k] = c->fp32_ok[pass][k];
  return QX_OK;
}

int qx_set_tensor_limit(qx_ctx* c, long long bytes) {
  if (!c || bytes < 0) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    QX_HIP(hipSetDevice(c->device));
    c->pairm_limit = (size_t)bytes;
    if (bytes > 0 && c->pairm_bytes > c->pairm_limit) drop_pairm(c);
    return QX_OK;
  });
}

int qx_set_streams(qx_ctx* c, int n) {
  if (!c || n < 1 || n > 8) return QX_EINVAL;
  c->nstreams = n;
  return QX_OK;
}

int qx_class_info(int cls, int* l4, int* nparts) {
  if (cls < 0 || cls >= QX_NUM_CLASSES) return QX_EINVAL;
  const QxClassEntry& e = qx_class_table[cls];
  if (l4) { l4[0] = e.la; l4[1] = e.lb; l4[2] = e.lc; l4[3] = e.ld; }
  if (nparts) *nparts = e.nparts;
  return QX_OK;
}

int qx_class_flops(int cls, double* eri, double* parts, int* ncomb) {
  if (cls < 0 || cls >= QX_NUM_CLASSES) return QX_EINVAL;
  const QxClassEntry& e = qx_class_table[cls];
  if (eri) *eri = e.eri_flops;
  for (int k = 0; k < e.nparts; ++k) {
    if (parts) parts[k] = e.part_flops[k];
    if (ncomb) ncomb[k] = e.part_ncomb[k];
  }
  return QX_OK;
}

int qx_max_parts(void) { return QX_DPARTS_CAP; }

int qx_class_jk(int cls, int* nparts, double* flops) {
  if (cls < 0 || cls >= QX_NUM_CLASSES) return QX_EINVAL;
  const QxClassEntry& e = qx_class_table[cls];
  if (nparts) *nparts = e.njk;
  for (int k = 0; k < e.njk; ++k)
    if (flops) flops[k] = e.jk_flops[k];
  return QX_OK;
}

int qx_class_groups(int cls, int* ngroups, double* flops, int* nparts) {
  if (cls < 0 || cls >= QX_NUM_CLASSES) return QX_EINVAL;
  const QxClassEntry& e = qx_class_table[cls];
  if (ngroups) *ngroups = e.ngroups;
  for (int k = 0; k < e.ngroups; ++k) {
    if (flops) flops[k] = e.group_flops[k];
    if (nparts) nparts[k] = e.group_parts[k];
  }
  return QX_OK;
}

int qx_class_quartets(const qx_ctx* c, long long* eri, long long* deri) {
  if (!c) return QX_EINVAL;
  for (int k = 0; k < QX_NUM_CLASSES; ++k) {
    if (eri) eri[k] = c->nq_class[k];
    if (deri) deri[k] = c->ndq_class[k];
  }
  return QX_OK;
}

int qx_profile_enable(qx_ctx* c, int on) {
  if (!c) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    if (!c->prof_pending.empty()) {
      const int rc = qx_profile_read(c, nullptr, nullptr, nullptr);
      if (rc != QX_OK) return rc;
    }
    c->profiling = on != 0;
    c->prof_ms.assign(QX_PROFILE_SLOTS, 0.0);
    c->prof_launches.assign(QX_PROFILE_SLOTS, 0);
    c->prof_pq.assign(QX_PROFILE_SLOTS, 0);
    return QX_OK;
  });
}

int qx_profile_read(qx_ctx* c, double* ms, long long* launches, long long* pq) {
  if (!c) return QX_EINVAL;
  return guarded(c, [&]() -> int {
    if (c->prof_ms.size() != QX_PROFILE_SLOTS) {
      c->prof_ms.assign(QX_PROFILE_SLOTS, 0.0);
      c->prof_launches.assign(QX_PROFILE_SLOTS, 0);
      c->prof_pq.assign(QX_PROFILE_SLOTS, 0);
    }
    for (auto& p : c->prof_pending) {
      QX_HIP(hipEventSynchronize(p.stop));
      float t = 0.0f;
      QX_HIP(hipEventElapsedTime(&t, p.start, p.stop));
      c->prof_ms[p.slot] += t;
      c->event_pool.push_back(p.start);
      c->event_pool.push_back(p.stop);
    }
    c->prof_pending.clear();
    for (int k = 0; k < QX_PROFILE_SLOTS; ++k) {
      if (ms) ms[k] = c->prof_ms[k];
      if (launches) launches[k] = c->prof_launches[k];
      if (pq) pq[k] = c->prof_pq[k];
    }
    return QX_OK;
  });
}

}  // extern "C"
