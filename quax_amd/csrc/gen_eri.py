"""Generates the per-angular-momentum-class ERI and ERI-derivative kernels.

One ERI kernel per canonical class (la lb | lc ld) with la >= lb, lc >= ld and
bra pair class >= ket pair class.  Each thread evaluates one primitive-pair
quartet (contracted shells are handled by summing primitive-pair quartets in
the epilogue), as straight-line code:

  1. setup (P, Q, W, rho) and the Boys function F_0..F_L,
  2. Obara-Saika vertical recurrence [e0|f0]^(m), emitted as SSA scalars in
     dependency order (bra side first, then transferred to the ket),
  3. Head-Gordon-Pople horizontal recurrence to (ab|cd), choosing the cheaper
     of bra-first / ket-first per class,
  4. an epilogue selected at run time (pair matrix, store, Schwarz diagonal) or
     the contraction of a K kernel.

Derivative kernels build d/dX_i (ab|cd) from d/dA_i phi_a = 2 alpha
phi_{a+1_i} - a_i phi_{a-1_i}.  Every kernel forms d/dA, d/dB, d/dC and
infers d/dD by translational invariance.  A class whose body would exceed
its node budget is split into parts over the Cartesian components of a
(then of b, then of c): each part evaluates only the output functions
(a, b, c, d) in its ranges.  A part recomputes the recurrence
nodes it shares with the others, but its live set fits the register file
(the unsplit heavy bodies spill several KB per lane to scratch, and scratch
latency, not arithmetic, then bounds them).  The heavy classes, and every
derivative tensor, use the quadrature kernels of qx_rys.h instead.

Usage: python gen_eri.py OUTDIR [LMAX] [--no-fp32]
"""
from __future__ import annotations

import json
import os
import sys

AX = "xyz"
# largest SSA node count allowed in one derivative body before it is split:
# a per-class table (picked by timing budget variants on the GPU), else
# DERIV_NODES; QX_DERIV_NODES in the environment overrides both (tuning builds)
DERIV_NODES = 2000
# the tuning tables (QX_TUNING_FILE names another file: tests, tuning builds)
_BUDGET_FILE = os.environ.get("QX_TUNING_FILE") or os.path.join(os.path.dirname(os.path.abspath(__file__)),
                                                                "deriv_budget.json")
DERIV_BUDGET = {}
if os.path.exists(_BUDGET_FILE):  # written by tune.py from GPU timings
    with open(_BUDGET_FILE) as _fh:
        DERIV_BUDGET = {tuple(int(ch) for ch in k): int(v) for k, v in json.load(_fh).get("budget", {}).items()}
_BUDGET_OVERRIDE = os.environ.get("QX_DERIV_NODES")
# waves per SIMD the adjoint kernels of a class are compiled for (0: the
# compiler's choice, one wave with 512 registers for the heavy classes);
# from the same tuning file, QX_GRAD_WAVES overrides (tuning builds)
DERIV_WAVES = {}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        DERIV_WAVES = {tuple(int(ch) for ch in k): int(v) for k, v in json.load(_fh).get("waves", {}).items()}
_WAVES_OVERRIDE = os.environ.get("QX_GRAD_WAVES")


DERIV_CSPLIT = {}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        DERIV_CSPLIT = {tuple(int(ch) for ch in k): int(v) for k, v in json.load(_fh).get("csplit", {}).items()}
_CSPLIT_OVERRIDE = os.environ.get("QX_CSPLIT")

# threads per block of the streaming J/K and gradient kernels per class
# (quartet tiles picked by tune.py --tiles from GPU timings; default 128)
TILES = {"jk": {}, "grad": {}}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        _t = json.load(_fh).get("tiles", {})
        TILES = {k: {tuple(int(ch) for ch in c): int(v) for c, v in _t.get(k, {}).items()} for k in ("jk", "grad")}

# classes whose adjoint-gradient kernels sum wave-uniform centres across the
# wavefront before the LDS accumulators (picked by tune.py --tiles)
GRAD_WAVE_REDUCE = {(0, 0, 0, 0), (1, 0, 0, 0), (1, 0, 1, 0), (1, 1, 0, 0), (2, 0, 0, 0)}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        _g = json.load(_fh).get("grad_wave_reduce")
        if _g is not None:
            GRAD_WAVE_REDUCE = {tuple(int(ch) for ch in c) for c in _g}

# copies of the gradient accumulators each class's adjoint blocks flush into
# (picked by tune.py --tiles; default 64)
GRAD_COPIES = {}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        GRAD_COPIES = {tuple(int(ch) for ch in c): int(v)
                       for c, v in json.load(_fh).get("grad_copies", {}).items()}

# classes whose mixed-precision passes may use FP32 (J/K, gradient): those
# whose FP32 kernels timed faster than their FP64 ones (fewer spills)
FP32_CLASSES = {"jk": set(), "grad": set()}
if os.path.exists(_BUDGET_FILE):
    with open(_BUDGET_FILE) as _fh:
        _f = json.load(_fh).get("fp32", {})
        FP32_CLASSES = {k: {tuple(int(ch) for ch in c) for c in _f.get(k, [])} for k in ("jk", "grad")}


def deriv_csplit(l):
    """c-component ranges per (a, b) part for classes whose (a, b) parts
    still exceed their budget (1 = no further split)."""
    if _CSPLIT_OVERRIDE:
        return int(_CSPLIT_OVERRIDE)
    return DERIV_CSPLIT.get(tuple(l), 1)


def deriv_waves(l):
    if _WAVES_OVERRIDE:
        return int(_WAVES_OVERRIDE)
    return DERIV_WAVES.get(tuple(l), 0)


def comps(l):
    out = []
    for i in range(l + 1):
        lx = l - i
        for j in range(i + 1):
            out.append((lx, i - j, j))
    return out


def ncart(l):
    return (l + 1) * (l + 2) // 2


def tot(v):
    return v[0] + v[1] + v[2]


def inc(v, i, d=1):
    w = list(v)
    w[i] += d
    return tuple(w)


def first_axis(v):
    for i in range(3):
        if v[i] > 0:
            return i
    return -1


Z3 = (0, 0, 0)


class VRR:
    """Obara-Saika vertical recurrence DAG for one primitive quartet."""

    def __init__(self):
        self.memo = {}
        self.lines = []
        self.nflop = 0

    def get(self, e, f, m):
        key = (e, f, m)
        if key in self.memo:
            return self.memo[key]
        if tot(f) > 0:
            i = first_axis(f)
            f1 = inc(f, i, -1)
            terms = [f"QC{AX[i]} * {self.get(e, f1, m)}", f"WQ{AX[i]} * {self.get(e, f1, m + 1)}"]
            self.nflop += 3
            if f1[i] > 0:
                f2 = inc(f1, i, -1)
                terms.append(f"R({f1[i]}) * oo2q * ({self.get(e, f2, m)} - rq * {self.get(e, f2, m + 1)})")
                self.nflop += 5
            if e[i] > 0:
                terms.append(f"R({e[i]}) * oo2pq * {self.get(inc(e, i, -1), f1, m + 1)}")
                self.nflop += 3
        elif tot(e) > 0:
            i = first_axis(e)
            e1 = inc(e, i, -1)
            terms = [f"PA{AX[i]} * {self.get(e1, Z3, m)}", f"WP{AX[i]} * {self.get(e1, Z3, m + 1)}"]
            self.nflop += 3
            if e1[i] > 0:
                e2 = inc(e1, i, -1)
                terms.append(f"R({e1[i]}) * oo2p * ({self.get(e2, Z3, m)} - rp * {self.get(e2, Z3, m + 1)})")
                self.nflop += 5
        else:
            name = f"b{m}"
            self.memo[key] = name
            return name
        name = f"v{len(self.memo)}"
        self.memo[key] = name
        self.lines.append(f"const R {name} = {' + '.join(terms)};")
        return name


class HRR:
    """Head-Gordon-Pople horizontal recurrence DAG.  order 'b' reduces b
    before d (so the ket HRR executes first), order 'd' the reverse."""

    def __init__(self, order):
        self.order = order
        self.memo = {}
        self.lines = []
        self.need = set()
        self.nflop = 0

    def get(self, a, b, c, d):
        key = (a, b, c, d)
        if key in self.memo:
            return self.memo[key]
        red_b = tot(b) > 0 and (self.order == "b" or tot(d) == 0)
        if red_b:
            i = first_axis(b)
            b1 = inc(b, i, -1)
            expr = f"{self.get(inc(a, i), b1, c, d)} + AB{AX[i]} * {self.get(a, b1, c, d)}"
            self.nflop += 2
        elif tot(d) > 0:
            i = first_axis(d)
            d1 = inc(d, i, -1)
            expr = f"{self.get(a, b, inc(c, i), d1)} + CD{AX[i]} * {self.get(a, b, c, d1)}"
            self.nflop += 2
        else:
            self.need.add((a, c))
            name = f"s_{a[0]}{a[1]}{a[2]}_{c[0]}{c[1]}{c[2]}"
            self.memo[key] = name
            return name
        name = f"h{len(self.memo)}"
        self.memo[key] = name
        self.lines.append(f"const R {name} = {expr};")
        return name


def build_dag(targets):
    """HRR + VRR DAG for the targets; also returns, per target, the number of
    HRR lines after which its value is available (emission is in target
    order, so consumers can be interleaved to keep live ranges short)."""
    best = None
    for order in "bd":
        h = HRR(order)
        outs, pos = [], []
        for t in targets:
            outs.append(h.get(*t))
            pos.append(len(h.lines))
        v = VRR()
        vn = {ac: v.get(ac[0], ac[1], 0) for ac in sorted(h.need)}
        cost = len(h.lines) + len(v.lines)
        if best is None or cost < best[0]:
            best = (cost, h, v, vn, outs, pos)
    return best[1:]


def interleave(hlines, groups):
    """groups: list of (position, [statements]) in non-decreasing position;
    returns HRR lines with each group's statements placed as soon as its
    inputs exist."""
    out = []
    gi = 0
    for i in range(len(hlines) + 1):
        while gi < len(groups) and groups[gi][0] <= i:
            out += groups[gi][1]
            gi += 1
        if i < len(hlines):
            out.append(hlines[i])
    return out


def emit_dblocks(L, nn):
    """Loads the six density blocks of the quartet (double) from A_.e.D into
    local arrays."""
    NA, NB, NC, ND = nn
    L.append("  const int n_ = A_.e.nbf;")
    L.append("  const double* Dm_ = A_.e.D;")
    L.append("  const int ia_ = A_.pr.bfa[P1], ib_ = A_.pr.bfb[P1], ic_ = A_.pr.bfa[P2], id_ = A_.pr.bfb[P2];")
    for nm, r0, nr, c0, nc in (("Dab", "ia_", NA, "ib_", NB), ("Dcd", "ic_", NC, "id_", ND),
                               ("Dac", "ia_", NA, "ic_", NC), ("Dad", "ia_", NA, "id_", ND),
                               ("Dbc", "ib_", NB, "ic_", NC), ("Dbd", "ib_", NB, "id_", ND)):
        L.append(f"  double {nm}[{nr * nc}];")
        L.append(f"  for (int r_ = 0; r_ < {nr}; ++r_) for (int c_ = 0; c_ < {nc}; ++c_) "
                 f"{nm}[r_ * {nc} + c_] = Dm_[({r0} + r_) * n_ + {c0} + c_];")


CENTRES = "ABCD"


def deriv_targets(l, part):
    """Targets of one derivative part, in emission order: for every
    (a,b,c,d) of the part's a/b ranges, for every (centre, x): raised, then
    lowered."""
    la, lb, lc, ld = l
    a0, a1 = part["a"]
    b0, b1 = part["b"]
    c0, c1 = part.get("c", (0, ncart(lc)))
    T = []
    for a in comps(la)[a0:a1]:
        for b in comps(lb)[b0:b1]:
            for c in comps(lc)[c0:c1]:
                for d in comps(ld):
                    for (cen, x) in part["combos"]:
                        q = [a, b, c, d]
                        k = CENTRES.index(cen)
                        up = list(q)
                        up[k] = inc(q[k], x)
                        T.append(tuple(up))
                        if q[k][x] > 0:
                            dn = list(q)
                            dn[k] = inc(q[k], x, -1)
                            T.append(tuple(dn))
    return T


def _classes(var, default):
    """Class set of a quadrature path; the environment overrides it (tuning builds)."""
    return set(os.environ.get(var, default).replace(",", " ").split())


# classes whose K, adjoint gradient and (stored) integrals come from the
# Rys-quadrature kernels (qx_rys.h) instead of the one-lane-per-quartet bodies.
# 280 functions, one lane / quadrature in us, all FP64: K 2110 183/797, 2111 283/308,
# 2120 299/412, 2210 119/373, 2220 350/289 (but 7.7/11.9 ms at 672 functions, where
# K' and density rows fill a CU's LDS and the quadrature has four wavefronts on it:
# the one-lane form stays, 0.06 ms slower at 280), 2121 829/288, 2211 530/228; gradient 1111 216/318, 2020 201/290, 2011 205/472,
# 2110 370/1608, and the split one-lane bodies of the listed classes 1.3 to 3
# times the quadrature's
RYS_K = _classes("QX_RYS_K", "2121 2211 2221 2222")
RYS_G = _classes("QX_RYS_G", "2111 2120 2121 2210 2211 2220 2221 2222")
RYS_E = _classes("QX_RYS_E", "2111 2120 2121 2211 2220 2221 2222")
# classes whose directional derivatives (K and adjoint gradient) are by quadrature.
# Gradient, one lane / quadrature in us, both in dual numbers: 196 functions 0000 42/493, 1010
# 157/1294, 1111 511/1219, 2011 302/1012, 2020 134/892, 2110 489/580, 2200 80/205;
# 12 atoms, minimal basis 0000 49/463, 1010 160/1143, 1110 117/1022, 1111 202/628;
# whole directional J/K pass 2.3/3.1 ms and 0.37/0.77 ms
RYS_H = _classes("QX_RYS_H", "2111 2120 2121 2210 2211 2220 2221 2222")


def _ranges(n, k):
    """k contiguous, nearly equal index ranges covering 0..n-1."""
    return [(i * n // k, (i + 1) * n // k) for i in range(k)]


def deriv_parts(l, budget=None):
    """Split the derivative of class l into kernels of at most `budget`
    recurrence nodes: whole class, else contiguous ranges of a components,
    else one a component with ranges of b components, else one (a, b) pair
    with ranges of c components (one (a, b, c) triple per part is the finest
    split)."""
    if budget is None:
        budget = int(_BUDGET_OVERRIDE) if _BUDGET_OVERRIDE else DERIV_BUDGET.get(tuple(l), DERIV_NODES)
    la, lb = l[0], l[1]
    NA, NB = ncart(la), ncart(lb)
    combos = [(c, x) for c in "ABC" for x in range(3)]

    NC = ncart(l[2])

    def part(ar, br, cr=(0, NC)):
        return {"combos": combos, "dinv": True, "a": ar, "b": br, "c": cr}

    def nodes(p):
        h, v, _, _, _ = build_dag(deriv_targets(l, p))
        return len(h.lines) + len(v.lines)

    whole = part((0, NA), (0, NB))
    if nodes(whole) <= budget:
        return [whole]
    for k in range(2, NA + 1):
        ps = [part(r, (0, NB)) for r in _ranges(NA, k)]
        if all(nodes(p) <= budget for p in ps):
            return ps
    for k in range(1, NB + 1):
        ps = [part((a, a + 1), r) for a in range(NA) for r in _ranges(NB, k)]
        if all(nodes(p) <= budget for p in ps):
            return ps
    # one (a, b) pair per part is still above the budget: c ranges, as many
    # as the class's csplit allows (1 keeps the (a, b) parts)
    kc = min(deriv_csplit(l), NC)
    return [part((a, a + 1), (b, b + 1), r) for a in range(NA) for b in range(NB) for r in _ranges(NC, kc)]


def emit_setup_tangent(L, Lt):
    """Set-up of a dual-number body: every geometric quantity is a qx_dual whose
    derivative part follows the atoms along A_.e.tv (exponents are fixed)."""
    L.append("  const double p = A_.pp.p[u1], q = A_.pp.p[u2];")
    L.append("  const QxTanPair tb_ = qx_tan_pair(A_, P1, u1), tk_ = qx_tan_pair(A_, P2, u2);")
    L.append("  const R Px = tb_.P[0], Py = tb_.P[1], Pz = tb_.P[2];")
    L.append("  const R Qx = tk_.P[0], Qy = tk_.P[1], Qz = tk_.P[2];")
    L.append("  const R Ax = tb_.A[0], Ay = tb_.A[1], Az = tb_.A[2];")
    L.append("  const R Cx = tk_.A[0], Cy = tk_.A[1], Cz = tk_.A[2];")
    L.append("  const R ABx = tb_.AB[0], ABy = tb_.AB[1], ABz = tb_.AB[2];")
    L.append("  const R CDx = tk_.AB[0], CDy = tk_.AB[1], CDz = tk_.AB[2];")
    L.append("  const double pq = p + q, opq = 1.0 / pq;")
    L.append("  const R Wx = (p * Px + q * Qx) * opq, Wy = (p * Py + q * Qy) * opq, Wz = (p * Pz + q * Qz) * opq;")
    L.append("  const R PQx = Px - Qx, PQy = Py - Qy, PQz = Pz - Qz;")
    L.append("  const double rho = p * q * opq;")
    L.append("  const R T = rho * (PQx * PQx + PQy * PQy + PQz * PQz);")
    L.append(f"  R F[{Lt + 1}];")
    L.append(f"  qx_boys_tan<{Lt}>(T, A_.boys, F);")
    L.append("  const R pref = (QX_TWO_PI_5_2 / (p * q * sqrt(pq))) * (tb_.K * tk_.K);")
    for m in range(Lt + 1):
        L.append(f"  const R b{m} = pref * F[{m}];")


def emit_setup(L, Lt, deriv_w):
    L.append("  const double p = A_.pp.p[u1], Kab = A_.pp.K[u1];")
    L.append("  const double Px = A_.pp.Px[u1], Py = A_.pp.Py[u1], Pz = A_.pp.Pz[u1];")
    L.append("  const double q = A_.pp.p[u2], Kcd = A_.pp.K[u2];")
    L.append("  const double Qx = A_.pp.Px[u2], Qy = A_.pp.Py[u2], Qz = A_.pp.Pz[u2];")
    L.append("  const double Ax = A_.pr.Ax[P1], Ay = A_.pr.Ay[P1], Az = A_.pr.Az[P1];")
    L.append("  const double Cx = A_.pr.Ax[P2], Cy = A_.pr.Ay[P2], Cz = A_.pr.Az[P2];")
    L.append("  const R ABx = (R)A_.pr.ABx[P1], ABy = (R)A_.pr.ABy[P1], ABz = (R)A_.pr.ABz[P1];")
    L.append("  const R CDx = (R)A_.pr.ABx[P2], CDy = (R)A_.pr.ABy[P2], CDz = (R)A_.pr.ABz[P2];")
    L.append("  const double pq = p + q, opq = 1.0 / pq;")
    L.append("  const double Wx = (p * Px + q * Qx) * opq, Wy = (p * Py + q * Qy) * opq, Wz = (p * Pz + q * Qz) * opq;")
    L.append("  const double PQx = Px - Qx, PQy = Py - Qy, PQz = Pz - Qz;")
    L.append("  const double rho = p * q * opq;")
    L.append("  const double T = rho * (PQx * PQx + PQy * PQy + PQz * PQz);")
    L.append(f"  double F[{Lt + 1}];")
    L.append(f"  qx_boys<{Lt}>(T, A_.boys, F);")
    L.append("  const double pref = QX_TWO_PI_5_2 * Kab * Kcd / (p * q * sqrt(pq));")
    for m in range(Lt + 1):
        L.append(f"  const R b{m} = (R)(pref * F[{m}]);")


def emit_vrr_consts(L, vrr_lines, S="R"):
    """S: type of the factors that depend on exponents alone."""
    used = "\n".join(vrr_lines)
    for ax in AX:
        if f"PA{ax}" in used:
            L.append(f"  const R PA{ax} = (R)(P{ax} - A{ax});")
        if f"WP{ax}" in used:
            L.append(f"  const R WP{ax} = (R)(W{ax} - P{ax});")
        if f"QC{ax}" in used:
            L.append(f"  const R QC{ax} = (R)(Q{ax} - C{ax});")
        if f"WQ{ax}" in used:
            L.append(f"  const R WQ{ax} = (R)(W{ax} - Q{ax});")
    if "oo2p " in used:
        L.append(f"  const {S} oo2p = ({S})(0.5 / p);")
    if "oo2q " in used:
        L.append(f"  const {S} oo2q = ({S})(0.5 / q);")
    if "oo2pq " in used:
        L.append(f"  const {S} oo2pq = ({S})(0.5 * opq);")
    if " rp " in used:
        L.append(f"  const {S} rp = ({S})(q * opq);")
    if " rq " in used:
        L.append(f"  const {S} rq = ({S})(p * opq);")


def _head(L, fn, sig, Lt, v, vn, ret="void", inline="__forceinline__", tangent=False):
    if tangent:
        L.append(f"__device__ {inline} {ret} {fn}(const QxArgs& A_, int P1, int P2, int u1, int u2{sig}) {{")
        L.append("  using R = qx_dual;")
        emit_setup_tangent(L, Lt)
        emit_vrr_consts(L, v.lines, "double")
        L += ["  " + x.replace("R(", "double(") for x in v.lines]
    else:
        L.append(f"template <typename R>\n__device__ {inline} {ret} {fn}(const QxArgs& A_, int P1, int P2, "
                 f"int u1, int u2{sig}) {{")
        emit_setup(L, Lt, False)
        emit_vrr_consts(L, v.lines)
        L += ["  " + x for x in v.lines]
    for (a, c), name in sorted(vn.items()):
        L.append(f"  const R s_{a[0]}{a[1]}{a[2]}_{c[0]}{c[1]}{c[2]} = {name};")


def emit_k_body(l, h, v, vn, outs, pos, tangent=False):
    """K body of a class (qx_kb_e*): the integrals of all primitives are summed
    as [e0|f0], then transferred and contracted with the density blocks one by
    one, all in FP64 also where the recursion is FP32 (summed in FP32, K of 49 x
    49 primitives was off by 2.7e-7 of its norm; rounded after the sum, 2.4e-8;
    rounded per primitive quartet only, 1.5e-9).  tangent: qx_kb_ve*, the same
    of the integrals' derivative along A_.e.tv."""
    NA, NB, NC, ND = (ncart(x) for x in l)
    N = NA * NB * NC * ND
    nm = "".join(map(str, l))
    S = "R" if tangent else "double"  # type of the sums and the transfer
    K = [f"template <typename R>\n__device__ __forceinline__ void qx_kb_{f've{nm}' if tangent else f'e{nm}_0'}(const QxArgs& A_, int P1, int P2, "
         f"int s_, int ns_, const double (&Dac)[{NA * NC}], const double (&Dad)[{NA * ND}], const double (&Dbc)[{NB * NC}], "
         f"const double (&Dbd)[{NB * ND}], double (&kac)[{NA * NC}], double (&kad)[{NA * ND}], "
         f"double (&kbc)[{NB * NC}], double (&kbd)[{NB * ND}]) {{"]
    names = {ac: f"s_{ac[0][0]}{ac[0][1]}{ac[0][2]}_{ac[1][0]}{ac[1][1]}{ac[1][2]}" for ac in sorted(vn)}
    K += [f"  {S} {x}(0.0);" for x in names.values()]
    K.append("  const int v1_ = A_.pr.pp_first[P1], v2_ = A_.pr.pp_first[P2], n2_ = A_.pr.pp_n[P2];")
    K.append("  for (int k_ = s_; k_ < A_.pr.pp_n[P1] * n2_; k_ += ns_) {")
    K.append("  const int u1 = v1_ + k_ / n2_, u2 = v2_ + k_ % n2_;")
    body = []
    if tangent:
        emit_setup_tangent(body, sum(l))
        emit_vrr_consts(body, v.lines, "double")
        body += ["  " + x.replace("R(", "double(") for x in v.lines]
    else:
        emit_setup(body, sum(l), False)
        emit_vrr_consts(body, v.lines)
        body += ["  " + x for x in v.lines]
    body = [x for x in body if not x.startswith(("  const R ABx", "  const R CDx"))]
    body += [f"  {names[ac]} += ({S}){vn[ac]};" for ac in sorted(vn)]
    K += ["  " + x for x in body] + ["  }"]
    if tangent:
        K.append("  const QxTanPair tb_ = qx_tan_pair(A_, P1, v1_), tk_ = qx_tan_pair(A_, P2, v2_);")
    for cd, pair, tan in (("AB", "P1", "tb_"), ("CD", "P2", "tk_")):
        K.append(f"  const {S} " + ", ".join(f"{cd}{ax} = {tan}.AB[{i}]" if tangent else f"{cd}{ax} = A_.pr.AB{ax}[{pair}]"
                                             for i, ax in enumerate(AX)) + ";")
    groups = []
    for k in range(N):
        i, rem = divmod(k, NB * NC * ND)
        j, rem = divmod(rem, NC * ND)
        kk, ll = divmod(rem, ND)
        ik, il, jk, jl = i * NC + kk, i * ND + ll, j * NC + kk, j * ND + ll
        groups.append((pos[k], [
            f"  {{ const double v_ = qx_value({outs[k]});",
            f"    kac[{ik}] += v_ * Dbd[{jl}]; kad[{il}] += v_ * Dbc[{jk}];",
            f"    kbc[{jk}] += v_ * Dad[{il}]; kbd[{jl}] += v_ * Dac[{ik}]; }}"]))
    hrr = [x.replace("const R ", f"const {S} ") for x in h.lines]
    K += ["  " + x if not x.startswith("  ") else x for x in interleave(hrr, groups)]
    K.append("}")
    return "\n".join(K)


def emit_eri_core(l):
    """Two bodies per class: qx_core_e* adds the integrals to an array (the
    pair-matrix / store / Schwarz epilogues), qx_kb_e* sums the primitive
    quartets of a contracted one and contracts each integral into the K'
    accumulators as soon as it is formed."""
    la, lb, lc, ld = l
    nn = (ncart(la), ncart(lb), ncart(lc), ncart(ld))
    NA, NB, NC, ND = nn
    N = NA * NB * NC * ND
    T = [(a, b, c, d) for a in comps(la) for b in comps(lb) for c in comps(lc) for d in comps(ld)]
    h, v, vn, outs, pos = build_dag(T)
    Lt = sum(l)
    nm = "".join(map(str, l))
    # array form
    L = []
    _head(L, f"qx_core_e{nm}", f", R (&o)[{N}]", Lt, v, vn)
    groups = [(pos[k], [f"  o[{k}] += {outs[k]};"]) for k in range(N)]
    L += ["  " + x if not x.startswith("  ") else x for x in interleave(h.lines, groups)]
    L.append("}")
    stats = dict(vrr=len(v.lines), vrr_flops=v.nflop, hrr=len(h.lines), hrr_flops=h.nflop, L=Lt, N=N,
                 flops=core_flops(Lt, v.nflop, h.nflop))
    K = emit_k_body(l, h, v, vn, outs, pos)
    # K epilogue: 4 fused multiply-adds per integral
    return "\n".join(L), [K], dict(stats, jk_flops=[core_flops(Lt, v.nflop, h.nflop) + 8 * N])


def emit_deriv_core(l, pi, part, tangent=False):
    """One derivative part: qx_gr_d* contracts each derivative integral with
    the density pair product as soon as it is formed (the adjoint gradient),
    so no derivative block is ever held whole.  tangent: qx_gt_d*, the same of
    the integrals' derivative along A_.e.tv."""
    la, lb, lc, ld = l
    nn = (ncart(la), ncart(lb), ncart(lc), ncart(ld))
    NA, NB, NC_, ND = nn
    N = NA * NB * NC_ * ND
    combos, dinv = part["combos"], part["dinv"]
    a0, a1 = part["a"]
    b0, b1 = part["b"]
    c0, c1 = part.get("c", (0, ncart(lc)))
    T = deriv_targets(l, part)
    h, v, vn, outs, pos = build_dag(T)
    Lt = sum(l) + 1
    nm = "".join(map(str, l))
    NC = len(combos)
    S = "double" if tangent else "R"  # factors without a derivative part
    wexpr = {"A": "A_.pp.a2[u1]", "B": "A_.pp.b2[u1]", "C": "A_.pp.a2[u2]", "D": "A_.pp.b2[u2]"}
    wdecl = [f"  const {S} w{c} = ({S}){wexpr[c]};" for c in sorted(set(cc for cc, _ in combos))]
    # per element: expressions of each combo and the position after which all exist
    elems = []
    ti = 0
    for ia, a in enumerate(comps(la)[a0:a1], a0):
        for ib, b in enumerate(comps(lb)[b0:b1], b0):
            for ic, c in enumerate(comps(lc)[c0:c1], c0):
                for id_, d in enumerate(comps(ld)):
                    e = ((ia * NB + ib) * NC_ + ic) * ND + id_
                    le = ((((ia - a0) * (b1 - b0) + (ib - b0)) * (c1 - c0)) + (ic - c0)) * ND + id_
                    q = [a, b, c, d]
                    exprs = []
                    last = 0
                    for ci, (cn, x) in enumerate(combos):
                        k = CENTRES.index(cn)
                        up = outs[ti]
                        last = max(last, pos[ti])
                        ti += 1
                        n = q[k][x]
                        dn = None
                        if n > 0:
                            dn = outs[ti]
                            last = max(last, pos[ti])
                            ti += 1
                        exprs.append(f"w{cn} * {up}" + (f" - {S}({n}) * {dn}" if dn else ""))
                    elems.append((e, le, last, exprs))
    # streaming adjoint form
    G = []
    _head(G, f"qx_{'gt' if tangent else 'gr'}_d{nm}_{pi}", f", double (&g)[{NC}]", Lt, v, vn, tangent=tangent)
    G += wdecl
    emit_dblocks(G, nn)
    groups = []
    for (e, le, last, exprs) in elems:
        i, rem = divmod(e, NB * NC_ * ND)
        j, rem = divmod(rem, NC_ * ND)
        kk, ll = divmod(rem, ND)
        ij, kl, ik, il, jk, jl = i * NB + j, kk * ND + ll, i * NC_ + kk, i * ND + ll, j * NC_ + kk, j * ND + ll
        st = [f"  {{ const double G_ = 2.0 * Dab[{ij}] * Dcd[{kl}] - 0.5 * (Dac[{ik}] * Dbd[{jl}] + "
              f"Dad[{il}] * Dbc[{jk}]);"]
        st += [f"    g[{ci}] += G_ * {'qx_value' if tangent else '(double)'}({ex});" for ci, ex in enumerate(exprs)]
        st.append("  }")
        groups.append((last, st))
    G += ["  " + x if not x.startswith("  ") else x for x in interleave(h.lines, groups)]
    G.append("}")
    cmask = sum(1 << CENTRES.index(c) for c in set(cc for cc, _ in combos))
    xmask = sum(1 << x for x in set(x for _, x in combos))
    nel = len(elems)
    stats = dict(part=pi, a=part["a"], b=part["b"], c=(c0, c1), dinv=dinv, vrr=len(v.lines), vrr_flops=v.nflop,
                 hrr=len(h.lines), hrr_flops=h.nflop, L=Lt, N=N, nel=nel, ncomb=NC,
                 flops=core_flops(Lt, v.nflop, h.nflop) + nel * (8 + 5 * NC))
    return "\n".join(G), stats, (cmask, xmask, dinv, NC)


def herm(L):
    """Hermite indices t + u + v <= L, v fastest (qx_herm's order)."""
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def j_cores(L1, L2s):
    """Per ket order L2 a body that runs the Hermite Coulomb recursion
    R^n_{t+1} = t R^{n+1}_{t-1} + X R^{n+1}_t and contracts it with the ket's
    Hermite density."""
    out = []
    for L2 in L2s:
        L = L1 + L2
        H1, H2 = herm(L1), herm(L2)
        S = [f"template <typename G, typename R>\n__device__ __forceinline__ void qx_jc_{L1}{L2}(R X, R Y, R Z, "
             f"const R (&b)[{L + 1}], const G (&h)[{len(H2)}], G (&j)[{len(H1)}]) {{"]
        memo = {}

        def r(t, n):
            if (t, n) in memo:
                return memo[(t, n)]
            if tot(t) == 0:
                name = f"b[{n}]"
            else:
                i = first_axis(t)
                t1 = inc(t, i, -1)
                ex = f"{'XYZ'[i]} * {r(t1, n + 1)}"
                if t1[i] > 0:
                    ex += f" + R({t1[i]}) * {r(inc(t1, i, -1), n + 1)}"
                name = f"r{len(memo)}"
                S.append(f"  const R {name} = {ex};")
            memo[(t, n)] = name
            return name

        for k, tau in enumerate(H2):
            for m, t in enumerate(H1):
                s = tuple(x + y for x, y in zip(t, tau))
                v = r(s, 0)
                if not v.startswith("b") and (s, "g") not in memo:
                    memo[(s, "g")] = v
                S.append(f"  j[{m}] += h[{k}] * G({v});")
        S.append("}")
        out += S + [""]
    return out


def emit_j(L1, outdir, lmax, fp32):
    """jeng_<L1>.hip, jengv_<L1>.hip: the J kernels of bra pairs of total
    angular momentum L1 (FP64 and FP32; dual numbers)."""
    cases = " ".join(f"QX_J_CASE({L1}, {L2})" for L2 in range(2 * lmax + 1))
    paths = []
    for name, last in (("jeng", f"QX_DEFINE_J_KERNEL({L1}, {1 if fp32 else 0}, {cases})"),
                       ("jengv", f"QX_DEFINE_JV_KERNEL({L1}, {cases})")):
        paths.append(os.path.join(outdir, f"{name}_{L1}.hip"))
        with open(paths[-1], "w") as fh:
            fh.write("\n".join(['#include "../qx_jk.h"', ""] + j_cores(L1, range(2 * lmax + 1)) + [last, ""]))
    return paths


def emit_small(outdir):
    """jk_small.hip: every K and J body of s and p shells in one kernel."""
    out = []
    for l in canonical_classes(1)[1]:
        nm = "".join(map(str, l))
        na, nb, nc, nd = map(ncart, l)
        out += emit_eri_core(l)[1] + [f"QX_DEFINE_K_BODY(e{nm}_0, {na}, {nb}, {nc}, {nd})", ""]
    for L1 in range(3):
        cases = " ".join(f"QX_J_CASE({L1}, {L2})" for L2 in range(3))
        out += j_cores(L1, range(3)) + [f"#define QX_SMALL_CASES_{L1} {cases}", ""]
    out.append("QX_DEFINE_SMALL()")
    path = os.path.join(outdir, "jk_small.hip")
    with open(path, "w") as fh:
        fh.write("\n".join(['#include "../qx_jk.h"', ""] + out + [""]))
    return path


def emit_small_grad(outdir):
    """grad_small.hip: every gradient body of s and p shells in one kernel;
    also the class of each of its lists."""
    out, cases, lists = [], [], []
    for ci, cls in enumerate(canonical_classes(1)[1]):
        nm = "".join(map(str, cls))
        for pi, part in enumerate(deriv_parts(cls)):
            out += [emit_deriv_core(cls, pi, part)[0], ""]
            cases += [f"    case {len(lists)}:",
                      "      qx_grad_block(A_, kl, b, sg, [&](int P1, int P2, int u1, int u2, double (&g)[QX_GRAD_NCOMB]) {",
                      f"        qx_gr_d{nm}_{pi}<double>(A_, P1, P2, u1, u2, g);", "      });", "      break;"]
            lists.append(ci)
    n = len(lists)
    out += [f"__constant__ int qx_small_class[{n}] = {{{', '.join(map(str, lists))}}};",
            "__global__ __launch_bounds__(QX_SMALL_BLOCK) void qx_small_grad(QxArgs A_, QxSmallGrad sm) {",
            "  __shared__ double sg[QX_GRAD_LDS];", "  const int w = blockIdx.x;", "  int i = 0;",
            f"  while (i < {n - 1} && w >= sm.end[i]) ++i;", "  const int at = w - (i ? sm.end[i - 1] : 0);",
            "  const QxKList& kl = sm.k[qx_small_class[i]];", "  QxKBlock b;",
            "  if (!qx_k_block(A_, kl, at % kl.nbra, at / kl.nbra, b)) return;", "  switch (i) {"] + cases + ["  }", "}",
            'extern "C" int qx_launch_small_grad(const QxArgs* a, const QxSmallGrad* sm, hipStream_t s) {',
            f"  if (sm->end[{n - 1}] <= 0) return 0;",
            f"  hipLaunchKernelGGL(qx_small_grad, dim3((unsigned)sm->end[{n - 1}]), dim3(QX_SMALL_BLOCK), 0, s, *a, *sm);",
            "  return (int)hipGetLastError();", "}"]
    path = os.path.join(outdir, "grad_small.hip")
    with open(path, "w") as fh:
        fh.write("\n".join(['#include "../qx_grad.h"', ""] + out + [""]))
    return path, lists


def emit_oei(la, lb, outdir):
    """oei_<la><lb>.hip: the attraction recurrences of one shell-pair class
    (the ERI bra recurrence with W - P = C - P and the (ss|ss) integrals
    replaced by the (s|1/r_C|s) ones) and its kernels (qx_oei.h)."""
    nm = f"{la}{lb}"
    A, B = comps(la), comps(lb)

    def head(L, v, PA="PA", PC="PC", nb=0):
        used = "\n".join(v.lines)
        for i, ax in enumerate(AX):
            if f"PA{ax}" in used:
                L.append(f"  const R PA{ax} = {PA}[{i}], WP{ax} = -{PC}[{i}];")
        if " rp " in used:
            L.append("  const double rp = 1.0;")
        for m in range(nb + 1):
            L.append(f"  const R b{m} = F[{m}];")
        L.extend("  " + x for x in v.lines)

    h, v, vn, outs, _ = build_dag([(a, b, Z3, Z3) for a in A for b in B])
    L = []
    L.append(f"#define NA_{nm} {len(A)}")
    L.append(f"#define NB_{nm} {len(B)}")
    L.append(f"template <typename R>\n__device__ __forceinline__ void qx_ov_{nm}(const R (&PA)[3], const R (&PC)[3], "
             f"double oo2p, const R (&F)[{la + lb + 1}], R (&s)[{len(vn)}]) {{")
    head(L, v, nb=la + lb)
    for k, (_, name) in enumerate(sorted(vn.items())):
        L.append(f"  s[{k}] += {name};")
    L.append("}")

    def hrr_in(L, vn, src=None):
        for k, ((a, c), name) in enumerate(sorted(vn.items())):
            L.append(f"  const R s_{a[0]}{a[1]}{a[2]}_000 = {f'{src}[{k}]' if src else name};")

    L.append(f"template <typename R>\n__device__ __forceinline__ void qx_ovh_{nm}(const R (&AB)[3], "
             f"const R (&s)[{len(vn)}], R (&o)[{len(A) * len(B)}]) {{")
    L.append("  const R ABx = AB[0], ABy = AB[1], ABz = AB[2];")
    hrr_in(L, vn, "s")
    L += ["  " + x for x in h.lines]
    L += [f"  o[{k}] = {x};" for k, x in enumerate(outs)]
    L.append("}")
    ns = len(vn)
    # derivative: d/dA and d/dB of every (a|b), contracted with the density block
    combos = [(c, x) for c in "AB" for x in range(3)]
    T, plan = [], []
    for i, a in enumerate(A):
        for j, b in enumerate(B):
            for ci, (cen, x) in enumerate(combos):
                q = [a, b]
                k = "AB".index(cen)
                up = list(q)
                up[k] = inc(q[k], x)
                T.append((up[0], up[1], Z3, Z3))
                n = q[k][x]
                if n > 0:
                    dn = list(q)
                    dn[k] = inc(q[k], x, -1)
                    T.append((dn[0], dn[1], Z3, Z3))
                plan.append((i * len(B) + j, ci, cen, n))
    h, v, vn, outs, pos = build_dag(T)
    L.append(f"template <typename R>\n__device__ __forceinline__ void qx_ovg_{nm}(const R (&PA)[3], const R (&PC)[3], "
             f"double oo2p, const R (&F)[{la + lb + 2}], const R (&AB)[3], double wA, double wB, "
             f"const double (&pd)[{len(A) * len(B)}], double (&g)[6]) {{")
    L.append("  const R ABx = AB[0], ABy = AB[1], ABz = AB[2];")
    head(L, v, nb=la + lb + 1)
    hrr_in(L, vn)
    groups, t = [], 0
    for (e, ci, cen, n) in plan:
        last, ex = pos[t], f"w{cen} * {outs[t]}"
        t += 1
        if n > 0:
            last, ex = max(last, pos[t]), ex + f" - double({n}) * {outs[t]}"
            t += 1
        groups.append((max(last, groups[-1][0] if groups else 0), [f"  g[{ci}] += pd[{e}] * oei_out({ex});"]))
    L += ["  " + x if not x.startswith("  ") else x for x in interleave(h.lines, groups)]
    L.append("}")
    L += ["", f"QX_DEFINE_OEI({nm}, {la}, {lb}, {ns})"]
    path = os.path.join(outdir, f"oei_{nm}.hip")
    with open(path, "w") as fh:
        fh.write("\n".join(['#include "../qx_oei.h"', ""] + L + [""]))
    return path


# Rys tables: must agree with qx_rys.h
RYS_TMAX, RYS_DEG, RYS_MAXN = 72, 12, 6


def rys_tables():
    """Roots and weights of exp(-T t^2) on [0, 1] in u = t^2, per order N <=
    RYS_MAXN and unit interval of T: degree-RYS_DEG polynomials in x in [-1, 1]
    (interpolation at Chebyshev nodes, monomial coefficients), then the
    half-range Hermite values that T scales for T >= RYS_TMAX.  The orthogonal
    polynomials come from Stieltjes' procedure on a 96-point Gauss-Legendre
    rule (Gautschi 1982), in long double throughout."""
    import numpy as np
    LD = np.longdouble
    one = LD(1)

    def legendre(n):
        x = np.polynomial.legendre.leggauss(n)[0].astype(LD)
        for last in (0, 0, 0, 1):
            p0, p1 = np.ones_like(x), x.copy()
            for k in range(2, n + 1):
                p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
            d = n * (x * p1 - p0) / (x * x - one)
            if not last:
                x = x - p1 / d
        return (x + one) / 2, one / ((one - x * x) * d * d)

    def gauss(u, w, N):
        """N-point Gauss rule of the discrete measure (u, w)."""
        a, b, nrm = [], [w.sum()], w.sum()
        pm, p = np.zeros_like(u), np.ones_like(u)
        for k in range(N):
            a.append((w * u * p * p).sum() / nrm)
            pm, p = p, (u - a[k]) * p - (b[k] * pm if k else 0)
            n2 = (w * p * p).sum()
            b.append(n2 / nrm)
            nrm = n2
        s = np.sqrt(np.array(b[1:N], float))
        r = np.linalg.eigvalsh(np.diag(np.array(a, float)) + np.diag(s, 1) + np.diag(s, -1)).astype(LD)
        for last in (0, 0, 0, 1):
            p0, p1 = np.zeros_like(r), np.ones_like(r)
            d0, d1 = np.zeros_like(r), np.zeros_like(r)
            S, nr = np.zeros_like(r), b[0]
            for k in range(N):
                S = S + p1 * p1 / nr
                nr = nr * b[k + 1]
                p0, p1, d0, d1 = (p1, (r - a[k]) * p1 - (b[k] * p0 if k else 0),
                                  d1, p1 + (r - a[k]) * d1 - (b[k] * d0 if k else 0))
            if not last:
                r = r - p1 / d1
        return np.concatenate([r, one / S])

    X, W = legendre(96)
    n = RYS_DEG + 1
    pi = LD("3.14159265358979323846264338327950288")
    th = (np.arange(n).astype(LD) + LD("0.5")) * pi / n
    # interpolation matrix: node values -> Chebyshev -> monomial coefficients
    cheb = np.array([[(one if j == 0 else LD(2)) / n * np.cos(j * t) for t in th] for j in range(n)])
    mono = np.zeros((n, n), LD)
    mono[0, 0] = mono[1, 1] = one
    for j in range(2, n):
        mono[j, 1:] = 2 * mono[j - 1, :-1]
        mono[j] -= mono[j - 2]
    M = mono.T @ cheb
    out = []
    for N in range(1, RYS_MAXN + 1):
        for iv in range(RYS_TMAX):
            F = np.array([gauss(X * X, W * np.exp(-(iv + (np.cos(t) + one) / 2) * X * X), N) for t in th])
            out += [(M @ F[:, f]) for f in range(2 * N)]
        # half-range Hermite: x^2 of exp(-x^2) on [0, inf) by mapping [0, 9]
        x, w = legendre(160)
        g = gauss((9 * x) ** 2, 9 * w * np.exp(-(9 * x) ** 2), N)
        out.append(g)
    flat = [v for c in out for v in c]
    return "// generated: Rys roots and weights\n" + ",\n".join(
        ", ".join(repr(float(v)) for v in flat[i:i + 8]) for i in range(0, len(flat), 8)) + "\n"


def core_flops(L, vrr_flops, hrr_flops):
    """Algorithmic FP operations of one primitive-quartet body (mul and add
    count 1, fused multiply-add 2): 30 for the pair/quartet setup, 12 + 4L
    for the Boys function (Taylor step plus downward recursion), then the
    recurrences as emitted."""
    return 30 + 12 + 4 * L + vrr_flops + hrr_flops


def canonical_classes(lmax):
    pairs = [(a, b) for a in range(lmax + 1) for b in range(a + 1)]
    out = []
    for i, (la, lb) in enumerate(pairs):
        for j, (lc, ld) in enumerate(pairs):
            if j <= i:
                out.append((la, lb, lc, ld))
    return pairs, out


# most derivative parts one adjoint-gradient launch (and source file) covers.
# Grouping several parts under blockIdx.y would fill the GPU for classes with
# few quartets, but hipcc's time on such a file grows far faster than the
# number of parts (12 (dd|dd) parts: 24 minutes inlined, 12 minutes as
# separate functions, against ~7 s per part alone), so every part keeps its
# own kernel (the launch table and ABI still speak of groups of one).
GROUP_PARTS = 1


def part_groups(nparts):
    """Contiguous, nearly equal groups of at most GROUP_PARTS parts."""
    ng = -(-nparts // GROUP_PARTS)
    return [list(range(i * nparts // ng, (i + 1) * nparts // ng)) for i in range(ng)]


def emit_class_files(cls, outdir, fp32):
    """Writes, per class: cls_<l>_e.hip (integrals: array-form kernel, or by
    quadrature for the heavy classes, whose array form would need 1 to 18 KB of
    scratch per lane), cls_<l>_j0.hip (K), cls_<l>_d0.hip (derivative slices), cls_<l>_v0.hip (directional
    derivatives of K and of the adjoint gradient) and cls_<l>_g<k>.hip (adjoint
    gradient: one kernel by quadrature, or one per derivative part)."""
    la, lb, lc, ld = cls
    nm = "".join(map(str, cls))
    dims = f"{ncart(la)}, {ncart(lb)}, {ncart(lc)}, {ncart(ld)}"
    N = ncart(la) * ncart(lb) * ncart(lc) * ncart(ld)
    files, stats = [], []

    def write(name, body, header="qx_device.h"):
        path = os.path.join(outdir, name)
        with open(path, "w") as fh:
            fh.write("\n".join([f'#include "../{header}"', ""] + body + [""]))
        files.append(path)

    src_e, jks, st = emit_eri_core(cls)
    if nm in RYS_E:
        write(f"cls_{nm}_e.hip", [f"QX_DEFINE_RYS_E(e{nm}, {la}, {lb}, {lc}, {ld})"], "qx_rys.h")
    else:
        write(f"cls_{nm}_e.hip", [src_e, "", f"QX_DEFINE_ERI_KERNEL(e{nm}, {N}, {dims})"], "qx_pairm.h")
    if nm in RYS_K:
        write(f"cls_{nm}_j0.hip", [f"QX_DEFINE_RYS_K(e{nm}_0, {la}, {lb}, {lc}, {ld}, {1 if fp32 else 0})"], "qx_rys.h")
    else:
        write(f"cls_{nm}_j0.hip", [jks[0], "", f"QX_DEFINE_K_KERNEL(e{nm}_0, {dims}, {1 if fp32 else 0})"], "qx_jk.h")
    stats.append((cls, "eri", st))
    write(f"cls_{nm}_d0.hip", [f"QX_DEFINE_RYS_D(d{nm}, {la}, {lb}, {lc}, {ld})"], "qx_rys.h")
    parts = deriv_parts(cls)
    if nm in RYS_H:
        hess = [f"QX_DEFINE_RYS_H(d{nm}, {la}, {lb}, {lc}, {ld})"]
    else:
        hess = []
        for pi, part in enumerate(parts):
            hess += [emit_deriv_core(cls, pi, part, tangent=True)[0], "",
                     f"__global__ __launch_bounds__(QX_BLOCK_MAX) void qx_kgv_d{nm}_{pi}(QxArgs A_, QxKList kl) {{",
                     "  __shared__ double sg[QX_GRAD_LDS];", "  QxKBlock b;", "  if (!qx_k_block(A_, kl, b)) return;",
                     "  qx_grad_block(A_, kl, b, sg, [&](int P1, int P2, int u1, int u2, double (&g)[QX_GRAD_NCOMB]) {",
                     f"    qx_gt_d{nm}_{pi}(A_, P1, P2, u1, u2, g);", "  });", "}"]
        kernels = ", ".join(f"qx_kgv_d{nm}_{pi}" for pi in range(len(parts)))
        hess.append(f"QX_DEFINE_GRADV_LAUNCHER(d{nm}, {kernels})")
    if nm in RYS_H:
        kv = [f"QX_DEFINE_RYS_KV(e{nm}, {la}, {lb}, {lc}, {ld})", ""]
    else:
        T = [(a, b, c, d) for a in comps(la) for b in comps(lb) for c in comps(lc) for d in comps(ld)]
        kv = [emit_k_body(cls, *build_dag(T), tangent=True), "", f"QX_DEFINE_KV_KERNEL(e{nm}, {dims})", ""]
    write(f"cls_{nm}_v0.hip", kv + hess, "qx_rys.h")
    gsrc = []
    for pi, part in enumerate(parts):
        src_g, st, (cmask, xmask, dinv, NC) = emit_deriv_core(cls, pi, part)
        assert (cmask, xmask, dinv, NC) == (7, 7, True, 9)
        gsrc.append(src_g)
        stats.append((cls, f"deriv{pi}", st))
    if nm in RYS_G:  # one kernel for the whole class
        groups = [list(range(len(parts)))]
        write(f"cls_{nm}_g0.hip", [f"QX_DEFINE_RYS_G(d{nm}_g0, {la}, {lb}, {lc}, {ld})"], "qx_rys.h")
        return files, stats, len(parts), groups
    groups = part_groups(len(parts))
    for gi, members in enumerate(groups):
        (pi,) = members
        w = deriv_waves(cls)
        attr = f" __attribute__((amdgpu_waves_per_eu({w}, {w})))" if w > 0 else ""
        kern = ["template <typename R>",
                f"__global__ __launch_bounds__(QX_BLOCK_MAX){attr} void qx_kg_d{nm}_g{gi}(QxArgs A_, QxKList kl) {{",
                "  __shared__ double sg[QX_GRAD_LDS];",
                "  QxKBlock b;",
                "  if (!qx_k_block(A_, kl, b)) return;",
                "  qx_grad_block(A_, kl, b, sg, [&](int P1, int P2, int u1, int u2, double (&g)[QX_GRAD_NCOMB]) {",
                f"    qx_gr_d{nm}_{pi}<R>(A_, P1, P2, u1, u2, g);", "  });", "}",
                f"QX_DEFINE_GRAD_LAUNCHER(d{nm}_g{gi}, {1 if fp32 else 0})"]
        write(f"cls_{nm}_g{gi}.hip", [gsrc[pi] for pi in members] + [""] + kern, "qx_grad.h")
    return files, stats, len(parts), groups


def main():
    outdir = sys.argv[1]
    lmax = int(sys.argv[2]) if len(sys.argv) > 2 else 2
    fp32 = "--no-fp32" not in sys.argv
    os.makedirs(outdir, exist_ok=True)
    _, classes = canonical_classes(lmax)
    files, allstats, nparts, flops, groups, jkf = [], [], {}, {}, {}, {}
    for cls in classes:
        f, s, np_, grp = emit_class_files(cls, outdir, fp32)
        files += f
        allstats += s
        nparts[cls] = np_
        groups[cls] = grp
        jkf[cls] = s[0][2]["jk_flops"]
        flops[cls] = (s[0][2]["flops"], [st["flops"] for _, _, st in s[1:]], [st["ncomb"] for _, _, st in s[1:]])
    pairs = [(a, b) for a in range(lmax + 1) for b in range(a + 1)]
    files += [emit_oei(a, b, outdir) for a, b in pairs]
    for L in range(2 * lmax + 1):
        files += emit_j(L, outdir, lmax, fp32)
    files.append(emit_small(outdir))
    path, small = emit_small_grad(outdir)
    files.append(path)
    with open(os.path.join(outdir, "qx_rys.inc"), "w") as fh:
        fh.write(rys_tables())
    D = ["// generated: kernel launch tables indexed by canonical class id", "#pragma once",
         f"#define QX_GEN_LMAX {lmax}", f"#define QX_NUM_CLASSES {len(classes)}",
         f"#define QX_MAX_DPARTS {max(nparts.values())}",
         f"#define QX_MAX_JKPARTS {max(len(v) for v in jkf.values())}",
         "static_assert(QX_MAX_JKPARTS <= QX_JKPARTS_CAP, \"J/K part table too small\");",
         "static_assert(QX_MAX_DPARTS <= QX_DPARTS_CAP, \"derivative part table too small\");", ""]
    for cls in classes:
        nm = "".join(map(str, cls))
        D.append(f'extern "C" int qx_launch_e{nm}(const QxArgs*, const QxLaunch*);')
        for pi in range(len(jkf[cls])):
            D.append(f'extern "C" int qx_launchj_e{nm}_{pi}(const QxArgs*, const QxLaunch*);')
        names = [f"qx_launch_d{nm}", f"qx_launchv_e{nm}", f"qx_launchh_d{nm}"]
        D += [f'extern "C" int {x}(const QxArgs*, const QxLaunch*);' for x in names]
        for gi in range(len(groups[cls])):
            D.append(f'extern "C" int qx_launchg_d{nm}_g{gi}(const QxArgs*, const QxLaunch*);')
    D.append("")
    D.append("static const QxClassEntry qx_class_table[QX_NUM_CLASSES] = {")
    for cls in classes:
        nm = "".join(map(str, cls))
        gl = ", ".join(f"qx_launchg_d{nm}_g{gi}" for gi in range(len(groups[cls])))
        ef, pf, pc = flops[cls]
        pfs = ", ".join(f"{x:.1f}" for x in pf)
        pcs = ", ".join(str(x) for x in pc)
        gfs = ", ".join(f"{sum(pf[p] for p in g):.1f}" for g in groups[cls])
        gps = ", ".join(str(len(g)) for g in groups[cls])
        jl = ", ".join(f"qx_launchj_e{nm}_{pi}" for pi in range(len(jkf[cls])))
        jfs = ", ".join(f"{x:.1f}" for x in jkf[cls])
        D.append(f"  {{{cls[0]}, {cls[1]}, {cls[2]}, {cls[3]}, qx_launch_e{nm}, qx_launch_d{nm}, qx_launchv_e{nm}, "
                 f"qx_launchh_d{nm}, {len(jkf[cls])}, {{{jl}}}, {{{jfs}}}, {nparts[cls]}, {len(groups[cls])}, {{{gl}}}, "
                 f"{ef:.1f}, {{{pfs}}}, {{{pcs}}}, {{{gfs}}}, {{{gps}}}}},")
    D.append("};")
    D.append("// per class: mixed-precision J/K and gradient passes may use FP32")
    D.append("static const unsigned char qx_fp32_default[QX_NUM_CLASSES][2] = {")
    for cls in classes:
        D.append(f"  {{{int(cls in FP32_CLASSES['jk'])}, {int(cls in FP32_CLASSES['grad'])}}},")
    D.append("};")
    D.append("// per class: the adjoint-gradient kernels reduce wave-uniform centres across the wavefront")
    D.append("static const unsigned char qx_gwred_default[QX_NUM_CLASSES] = {")
    D.append("  " + ", ".join(str(int(cls in GRAD_WAVE_REDUCE)) for cls in classes))
    D.append("};")
    D.append("// per class: copies of the gradient accumulators its adjoint blocks flush into")
    D.append("static const int qx_gcopy_default[QX_NUM_CLASSES] = {")
    D.append("  " + ", ".join(str(GRAD_COPIES.get(cls, 64)) for cls in classes))
    D.append("};")
    D.append("// per class: threads per block of the streaming J/K and gradient kernels")
    D.append("static const int qx_tile_default[QX_NUM_CLASSES][2] = {")
    for cls in classes:
        D.append(f"  {{{TILES['jk'].get(cls, 128)}, {TILES['grad'].get(cls, 128)}}},")
    D.append("};")
    D.append("// J kernels per bra pair angular momentum")
    D += [f'extern "C" int qx_launch_jeng_{L}(const QxArgs*, const QxJList*, int, int, int, hipStream_t);'
          for L in range(2 * lmax + 1)]
    D.append(f"static int (*const qx_j_table[{2 * lmax + 1}])(const QxArgs*, const QxJList*, int, int, int, hipStream_t) = {{"
             + ", ".join(f"qx_launch_jeng_{L}" for L in range(2 * lmax + 1)) + "};")
    for name, table, what in (("k", RYS_K, "K"), ("g", RYS_G, "the adjoint gradient"),
                              ("h", RYS_H, "the directional derivatives of K and of the adjoint gradient")):
        D.append(f"// per class: {what} by Rys quadrature")
        D.append(f"static const unsigned char qx_rys_{name}[QX_NUM_CLASSES] = {{")
        D.append("  " + ", ".join(str(int("".join(map(str, cls)) in table)) for cls in classes))
        D.append("};")
    D.append('extern "C" int qx_launch_small_grad(const QxArgs*, const QxSmallGrad*, hipStream_t);')
    D.append(f"static const int qx_small_grad_class[{len(small)}] = {{{', '.join(map(str, small))}}};")
    D.append(f"#define QX_SMALL_GRADS {len(small)}")
    D.append('extern "C" int qx_launch_small(const QxArgs*, const QxSmall*, unsigned, hipStream_t);')
    D.append("// one-electron kernels per shell-pair class")
    D += [f'extern "C" int qx_launch_oei_{a}{b}(const QxOei*, int, hipStream_t);' for a, b in pairs]
    D.append(f"static int (*const qx_oei_table[{len(pairs)}])(const QxOei*, int, hipStream_t) = {{"
             + ", ".join(f"qx_launch_oei_{a}{b}" for a, b in pairs) + "};")
    with open(os.path.join(outdir, "qx_classes.inc"), "w") as fh:
        fh.write("\n".join(D) + "\n")
    with open(os.path.join(outdir, "stats.txt"), "w") as fh:
        for cls, kind, st in allstats:
            fh.write(f"{cls} {kind} {st}\n")
    print("\n".join(files))


if __name__ == "__main__":
    main()
