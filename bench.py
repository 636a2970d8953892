#!/usr/bin/env python
"""ERI + dERI shell-quartet throughput on one MI355X.

Workload (default): the 10-atom synthetic cluster (6 C + 4 H, seeded, 8-bohr
cube, minimum separation 1.8 bohr), even-tempered spherical basis (280 AO /
300 Cartesian functions), Schwarz threshold 1e-12, FP64.  One step is one
pass of the hot path over the whole molecule:

  * the ERI pass: every canonical screened shell quartet, contracted with the
    density into J and K (integral-direct Fock build), and
  * the dERI pass: every canonical screened quartet not on a single atom,
    differentiated and contracted with the density pair products (adjoint
    HF gradient, two-electron part).

The density is the converged RHF density of the same molecule (SCF run
before the timed region).  value = (ERI quartets + dERI quartets) / step
time, inputs resident in HBM.  The HF energy + gradient wall time is reported
beside it.

Prints ONE JSON line (rank 0).  --gpus above 1 is refused: this build runs on
one GPU.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "ERI+dERI shell-quartets/s; HF-gradient wall time, mixed vs FP64 @1e-8 Eh"
PEAK_FP64 = 78.6e12     # MI355X FP64 (vector and matrix) peak, FLOP/s
PEAK_HBM = 8.0e12       # bytes/s


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def kernel_table(eng):
    """Per profile slot: kernel name and algorithmic flops per primitive
    quartet (including the epilogue contraction)."""
    import ctypes
    from quax_amd.csrc import gen_eri  # which classes run by quadrature
    L = eng.L
    ncart = lambda l: (l + 1) * (l + 2) // 2
    classes = {}
    info = {}
    for slot in range(L.qx_profile_slots()):
        kind, cls, part, f32 = (ctypes.c_int() for _ in range(4))
        L.qx_profile_slot(slot, ctypes.byref(kind), ctypes.byref(cls), ctypes.byref(part), ctypes.byref(f32))
        c = cls.value
        if c not in classes:
            l4 = (ctypes.c_int * 4)()
            npart = ctypes.c_int()
            L.qx_class_info(c, l4, ctypes.byref(npart))
            ef = ctypes.c_double()
            pf = (ctypes.c_double * L.qx_max_parts())()
            pc = (ctypes.c_int * L.qx_max_parts())()
            L.qx_class_flops(c, ctypes.byref(ef), pf, pc)
            ngr = ctypes.c_int()
            gf = (ctypes.c_double * L.qx_max_parts())()
            gp = (ctypes.c_int * L.qx_max_parts())()
            L.qx_class_groups(c, ctypes.byref(ngr), gf, gp)
            njk = ctypes.c_int()
            jf = (ctypes.c_double * 8)()
            L.qx_class_jk(c, ctypes.byref(njk), jf)
            classes[c] = (tuple(l4), ngr.value, ef.value, list(gf), njk.value, list(jf))
        # derivative slots of the gradient pass are per group of parts
        l4, npart, ef, pf, njk, jf = classes[c]
        nm = "".join(map(str, l4))
        tp = "float" if f32.value else "double"
        N = ncart(l4[0]) * ncart(l4[1]) * ncart(l4[2]) * ncart(l4[3])
        key = ("eri", "deriv", "jk")[kind.value] + ("32" if f32.value else "64")
        if kind.value == 0:
            info[slot] = (f"qx_k_e{nm}<{tp}>", ef, nm, key)
        elif kind.value == 2:
            # part 0: K of the class; part 1: J of the bra pairs (la, lb), booked under (la lb|la lb)
            args = ", ".join(map(str, l4))
            name = f"qx_rk<{args}, {tp}>" if nm in gen_eri.RYS_K else f"qx_kk_e{nm}_{part.value}<{tp}>"
            if part.value:
                name = f"qx_jeng_{l4[0] + l4[1]}<{tp}>"
            info[slot] = (name, jf[part.value] if part.value < njk else 0.0, nm, key)
        elif part.value < npart:
            name = f"qx_rg<{', '.join(map(str, l4))}>" if nm in gen_eri.RYS_G else f"qx_kg_d{nm}_g{part.value}<{tp}>"
            info[slot] = (name, pf[part.value], nm, key)
        else:
            info[slot] = (f"unused slot {slot}", 0.0, nm, key)
    return info


def flop_model():
    """Algorithmic FLOPs per canonical quartet and class (textbook HGP
    counts of the whole class, quax_amd/csrc/flop_model.json)."""
    with open(os.path.join(ROOT, "quax_amd", "csrc", "flop_model.json")) as fh:
        return json.load(fh)["classes"]


def slot_algorithmic_flops(table, model, eng, slot):
    """Algorithmic FLOPs per primitive quartet that one launch in `slot`
    accounts for: the class's J/K count for a J/K kernel; for one part of a
    split derivative class, the class's adjoint count shared out over its
    parts in proportion to their executed counts."""
    import ctypes
    name, fl, nm, key = table[slot]
    if key.startswith("jk"):
        njk = ctypes.c_int()
        jf = (ctypes.c_double * 8)()
        cls = [k for k in range(eng.L.qx_num_classes()) if table_class_name(eng, k) == nm][0]
        eng.L.qx_class_jk(cls, ctypes.byref(njk), jf)
        return model[nm]["jk"] * fl / sum(jf[:njk.value])
    if key.startswith("deriv"):
        cls = [k for k in range(eng.L.qx_num_classes()) if table_class_name(eng, k) == nm][0]
        ngr = ctypes.c_int()
        gf = (ctypes.c_double * eng.L.qx_max_parts())()
        gp = (ctypes.c_int * eng.L.qx_max_parts())()
        eng.L.qx_class_groups(cls, ctypes.byref(ngr), gf, gp)
        return model[nm]["adjoint"] * fl / sum(gf[:ngr.value])
    return model[nm]["eri"]


def table_class_name(eng, cls):
    import ctypes
    l4 = (ctypes.c_int * 4)()
    npart = ctypes.c_int()
    eng.L.qx_class_info(cls, l4, ctypes.byref(npart))
    return "".join(map(str, l4))


def host_cpu():
    """(logical CPUs, model name) of this host."""
    model = ""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return os.cpu_count() or 1, model


def measured_traffic(workload, kernel):
    """HBM bytes per launch that counter runs recorded for this kernel on this
    workload (profiles/hbm_traffic.txt), else None."""
    path = os.path.join(ROOT, "profiles", "hbm_traffic.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        f = line.split()  # workload, kernel (template arguments hold blanks), bytes
        if len(f) >= 3 and not line.startswith("#") and f[0] == workload and " ".join(f[1:-1]) == kernel:
            return float(f[-1])
    return None


def class_times(table, ms, steps):
    """Kernel ms per step summed per class: {class: {jk64, deriv64, ...}}."""
    out = {}
    for k, t in enumerate(ms):
        if t > 0:
            _, _, nm, key = table[k]
            out.setdefault(nm, {})
            out[nm][key] = out[nm].get(key, 0.0) + float(t) / steps
    return out


def class_roofline(eng, model, times):
    """Per class, one stream: quartets of the J/K and adjoint passes,
    algorithmic GFLOP per pass (the FLOP model's per-quartet counts) and the
    TFLOP/s its FP64 kernels reach."""
    out = {}
    for l4, ne, nd, _ in eng.class_quartets():
        nm = "".join(map(str, l4))
        t = times.get(nm, {})
        jk_ms, gr_ms = t.get("jk64", 0.0), t.get("deriv64", 0.0)
        gj, gg = model[nm]["jk"] * ne / 1e9, model[nm]["adjoint"] * nd / 1e9
        out[nm] = {"jk_quartets": int(ne), "grad_quartets": int(nd), "jk_gflop": gj, "grad_gflop": gg,
                   "jk_ms": jk_ms, "grad_ms": gr_ms,
                   "jk_tflops": gj / jk_ms if jk_ms > 0 else None,
                   "grad_tflops": gg / gr_ms if gr_ms > 0 else None}
    return out


def cpu_baseline(mol, basis, tol, eng, seconds):
    """Times the CPU oracle (C restatement of the reference's quartet loop
    and of the Libint HGP arithmetic) on a seeded uniform sample of the same
    canonical screened quartets, ERI and first-derivative, with OpenMP."""
    import numpy as np
    import oracle
    ob = oracle.OracleBasis(mol, basis)
    vals, pairs = eng.schwarz_screening()
    l = np.array([s.l for s in basis.shells])
    atom = np.array([s.atom for s in basis.shells])
    # canonical pair order as the device builds it: class, then Schwarz desc
    p = pairs
    la, lb = l[p[:, 0]], l[p[:, 1]]
    a = np.where(la >= lb, p[:, 0], p[:, 1])
    b = np.where(la >= lb, p[:, 1], p[:, 0])
    cls = l[a] * (l[a] + 1) // 2 + l[b]
    Q = vals[p[:, 0], p[:, 1]]
    order = np.lexsort((-Q, cls))
    a, b, cls, Q = a[order], b[order], cls[order], Q[order]
    rng = np.random.default_rng(11)
    # sample bra pairs proportionally to their admissible ket counts
    tol2 = tol * tol
    counts = np.zeros(len(a), dtype=np.int64)
    ket_lists = {}
    for X in np.unique(cls):
        for Y in np.unique(cls):
            if Y > X:
                continue
            bi = np.where(cls == X)[0]
            ki = np.where(cls == Y)[0]
            kq = Q[ki]
            for ii, i in enumerate(bi):
                kc = int(np.searchsorted(-kq, -tol2 / Q[i], side="right")) if Q[i] > 0 else 0
                if X == Y:
                    kc = min(kc, ii + 1)
                counts[i] += kc
                ket_lists.setdefault(i, []).append((ki, kc))
    total = counts.sum()
    # the host cores one GPU's job may use here: OMP_NUM_THREADS is that
    # share (16 per GPU on the MI355X hosts), else every logical CPU
    nthreads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or (os.cpu_count() or 1)

    cum = np.cumsum(counts)

    def sample(n, deriv):
        out = []
        while len(out) < n:
            t = int(rng.integers(total))
            i = int(np.searchsorted(cum, t, side="right"))
            r = t - (cum[i - 1] if i > 0 else 0)
            for ki, kc in ket_lists[i]:
                if r < kc:
                    j = ki[r]
                    break
                r -= kc
            q = (a[i], b[i], a[j], b[j])
            if deriv and len({atom[s] for s in q}) == 1:
                continue
            out.append(q)
        return np.array(out, dtype=np.int32)

    res = {}
    for deriv in (False, True):
        n = 2000
        while True:
            qs = sample(n, deriv)
            t0 = time.perf_counter()
            ob.quartet_batch(qs, nthreads=nthreads, deriv=deriv)
            dt = time.perf_counter() - t0
            if dt > seconds / 2 or n >= 2_000_000:
                break
            n = int(n * min(20.0, max(2.0, (seconds / 2) / max(dt, 1e-3))))
        res["deri" if deriv else "eri"] = (len(qs) / dt, len(qs), dt)
    return res, nthreads


def hf_energy_gradient(eng, mol, precision, thr, graph=False):
    """RHF energy (DIIS, conv 1e-10) + analytic gradient; wall times.
    graph: SCF iterations replayed from one captured HIP graph."""
    import torch
    from quax_amd.methods.hartree_fock import restricted_hartree_fock, rhf_gradient
    opts = {"diis": True, "spectral_shift": False, "conv": 1e-10, "maxit": 200, "precision": precision,
            "fp32_threshold": thr, "graph": graph}
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    E, aux = restricted_hartree_fock(eng, mol.nelectron(), opts, return_aux_data=True)
    torch.cuda.synchronize()
    t_scf = time.perf_counter() - t0
    t0 = time.perf_counter()
    grad = rhf_gradient(eng, aux, precision=precision, fp32_threshold=thr)
    torch.cuda.synchronize()
    return E, aux, grad, t_scf, time.perf_counter() - t0


def hf_mixed_vs_fp64(workload_mol, thr):
    """RHF energy + analytic gradient wall time of one molecule, FP64 and
    mixed (FP32 recursion below the Schwarz-bound threshold), with the mixed
    run's energy and gradient error against FP64."""
    import numpy as np
    from quax_amd.basis import BasisSet
    from quax_amd.engine import EriEngine
    mol = workload_mol
    basis = BasisSet.build(mol, "even-tempered", pure=True)
    with EriEngine(mol, basis, ints_tol=1e-12) as eng:
        n64, n32 = eng.mixed_quartets(thr)
        S0, _, _ = eng.oei()
        for prec in (0, 1):
            eng.jk(S0, precision=prec, fp32_threshold=thr)
            eng.eri_grad(S0, precision=prec, fp32_threshold=thr)
        E, aux, g, ts, tg = hf_energy_gradient(eng, mol, "fp64", thr)
        Em, auxm, gm, tsm, tgm = hf_energy_gradient(eng, mol, "mixed", thr)
    log(f"[bench] {mol.natom()} atoms ({basis.nbf()} AO): FP64 HF energy + gradient {ts + tg:.2f} s "
        f"({aux['iterations']} it), mixed @ {thr:g} {tsm + tgm:.2f} s ({auxm['iterations']} it), "
        f"dE {Em - E:.2e}, max dg {np.abs(gm - g).max():.2e}")
    return {"natom": mol.natom(), "nbf": basis.nbf(), "fp32_threshold": thr,
            "fp32_quartet_fraction": n32 / max(n64 + n32, 1),
            "hf_gradient_wall_s_fp64": ts + tg, "hf_gradient_wall_s_mixed": tsm + tgm,
            "scf_iterations_fp64": aux["iterations"], "scf_iterations_mixed": auxm["iterations"],
            "energy_error_mixed": Em - E, "grad_max_error_mixed": float(np.abs(gm - g).max()),
            "speedup_mixed": (ts + tg) / (tsm + tgm)}


def timed_steps(eng, D, steps, warmup, precision, thr, profile):
    """warmup + steps of (J/K pass, adjoint gradient pass); returns seconds
    and, when profile is set, the per-slot HIP-event kernel times."""
    import torch
    J = torch.empty_like(D)
    K = torch.empty_like(D)

    def step():
        eng.jk(D, precision=precision, fp32_threshold=thr, out=(J, K))
        eng.eri_grad(D, precision=precision, fp32_threshold=thr)

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    if profile:
        eng.profile(True)
    t0 = time.perf_counter()
    for i in range(steps):
        step()
        log(f"[bench] {'fp64' if precision == 0 else 'mixed'} step {i + 1}/{steps}")
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    prof = None
    if profile:
        prof = eng.profile_read()
        eng.profile(False)
    return dt, prof


def bench_batch(args):
    """Batched RHF energy + analytic gradient of the first --batch-size
    molecules of the seeded 256-molecule set (3-12 atoms, C/H/O), FP64: each
    chunk of --chunk molecules is one integral context with the molecules as
    fragments, its SCF iterations replayed from one captured HIP graph
    (converged molecules masked out of J/K), then one adjoint-gradient pass;
    the first three molecules are checked against single-molecule runs."""
    import numpy as np
    import torch
    from quax_amd import workloads
    from quax_amd.basis import BasisSet
    from quax_amd.engine import EriEngine
    from quax_amd.methods.batch import batched_rhf
    from quax_amd.methods.hartree_fock import restricted_hartree_fock, rhf_gradient
    mols = workloads.batch256()[:args.batch_size]
    graph = not args.no_graph
    batched_rhf(mols[:2], "even-tempered", pure=True, ints_tol=1e-12, conv=1e-6, graph=graph)   # warm-up
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    E, G, aux = [], [], {"iterations": [], "converged": [], "nbf": []}
    for c0 in range(0, len(mols), args.chunk):
        Ec, Gc, ac = batched_rhf(mols[c0:c0 + args.chunk], "even-tempered", pure=True, ints_tol=1e-12, conv=1e-10,
                                 maxit=args.maxit, graph=graph)
        E += Ec
        G += Gc
        for k in ("iterations", "converged", "nbf"):
            aux[k] += ac[k]
        log(f"[bench] batch molecules {c0}-{c0 + len(Ec) - 1}: {time.perf_counter() - t0:.1f} s so far, "
            f"iterations max {max(ac['iterations'])}, converged {sum(ac['converged'])}/{len(Ec)}"
            + f"; setup {ac['setup_s']:.1f} s, SCF {ac['scf_s']:.1f} s"
            + (f" (graph {ac['graph_s']:.1f} s, {ac['stalled']} finished eagerly)" if "graph_s" in ac else "")
            + f", gradient {ac['finish_s']:.1f} s (ERI part {ac.get('eri_grad_s', 0.0):.1f} s)")
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    # per-molecule check against single-molecule eager runs (the first
    # --check molecules); molecules that either SCF needs more than 40
    # iterations for have several stationary states that DIIS reaches along
    # rounding-dependent paths, so they are counted but not compared
    errs, unsettled = [], 0
    t1 = time.perf_counter()
    nchk = min(args.check, len(mols))
    for k in range(nchk):
        b = BasisSet.build(mols[k], "even-tempered", pure=True)
        with EriEngine(mols[k], b, ints_tol=1e-12) as e1:
            Ek, auxk = restricted_hartree_fock(e1, mols[k].nelectron(), {"diis": True, "spectral_shift": False,
                                                                        "conv": 1e-10, "maxit": args.maxit},
                                               return_aux_data=True)
            gk = rhf_gradient(e1, auxk)
        if auxk["iterations"] > 40 or aux["iterations"][k] > 40 or auxk["drms"] > 1e-10 or not aux["converged"][k]:
            unsettled += 1
            continue
        errs.append((abs(E[k] - Ek), float(np.abs(G[k] - gk).max())))
    torch.cuda.synchronize()
    single = (time.perf_counter() - t1) / nchk if nchk else None
    out = {"metric": "batched RHF energy + gradient, molecules/s", "value": len(mols) / wall,
           "unit": "molecules/s", "n_gpus": 1, "higher_is_better": True, "dtype": "f64", "data": "synthetic",
           "config": {"workload": f"first {len(mols)} of 256 seeded molecules (3-12 atoms, C/H/O 0.4/0.4/0.2), "
                                  f"even-tempered spherical basis, {sum(aux['nbf'])} AO total, Schwarz 1e-12, "
                                  "conv 1e-10",
                      "chunk": args.chunk, "graph_scf": graph, "maxit": args.maxit,
                      "wall_s": wall, "iterations_max": max(aux["iterations"]),
                      "all_converged": all(aux["converged"]),
                      "converged": int(sum(aux["converged"])),
                      "single_molecule_s_each": single,
                      "speedup_vs_single": len(mols) / wall * single if single else None,
                      "checked_vs_single": len(errs), "unsettled_in_check": unsettled,
                      "max_energy_error_vs_single": max((e for e, _ in errs), default=None),
                      "max_grad_error_vs_single": max((g for _, g in errs), default=None)}}
    print(json.dumps(out), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--cpu-seconds", type=float, default=20.0, help="CPU baseline budget (0 = skip)")
    ap.add_argument("--workload", default="cluster10", choices=["cluster10", "cluster24", "water", "batch"])
    ap.add_argument("--batch-size", type=int, default=32,
                    help="batch workload: molecules of the seeded 256-molecule set")
    ap.add_argument("--chunk", type=int, default=32, help="batch workload: molecules per context and graph")
    ap.add_argument("--no-graph", action="store_true", help="batch workload: host-driven lock-step SCF")
    ap.add_argument("--check", type=int, default=8, help="batch workload: molecules checked against single runs")
    ap.add_argument("--maxit", type=int, default=100,
                    help="batch workload: SCF iteration cap (100 is the reference's default, core.py:34)")
    ap.add_argument("--fp32-threshold", type=float, default=1e-8,
                    help="Schwarz bound below which the mixed runs use FP32 quartets")
    ap.add_argument("--streams", type=int, default=4, help="streams per pass (1 = every kernel timed alone)")
    ap.add_argument("--no-scf", action="store_true",
                    help="skip the SCF and use the core-Hamiltonian density (profiling runs)")
    ap.add_argument("--sweep", default="",
                    help="comma-separated FP32 thresholds: mixed HF energy + gradient error and time at each")
    ap.add_argument("--no-mixed", action="store_true", help="skip every mixed-precision run (FP64-only builds)")
    ap.add_argument("--no-cluster24", action="store_true",
                    help="skip the 24-atom mixed-vs-FP64 HF energy + gradient timing")
    ap.add_argument("--copy-probe", action="store_true",
                    help="also run a plain 512 MiB device copy (HBM-counter calibration for profiler runs)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py: this build runs on one GPU; --gpus must be 1 (multi-GPU sharding is design-only)",
              file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    from quax_amd import workloads
    from quax_amd.basis import BasisSet
    from quax_amd.engine import EriEngine

    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)
    tol = 1e-12
    thr = args.fp32_threshold
    if args.workload == "batch":
        return bench_batch(args)
    if args.workload == "water":
        mol, bname, pure = workloads.water_sto3g(), "sto-3g", False
    elif args.workload == "cluster24":
        mol, bname, pure = workloads.cluster24(), "even-tempered", True
    else:
        mol, bname, pure = workloads.cluster10(), "even-tempered", True
    basis = BasisSet.build(mol, bname, pure=pure)
    t_init = time.perf_counter()
    eng = EriEngine(mol, basis, ints_tol=tol)
    eng.set_streams(args.streams)
    torch.cuda.synchronize()
    t_init = time.perf_counter() - t_init
    cq = eng.class_quartets()
    q_eri = int(sum(x[1] for x in cq))
    q_deri = int(sum(x[2] for x in cq))
    n64, n32 = eng.mixed_quartets(thr) if not args.no_mixed else (q_eri, 0)
    log(f"[bench] {args.workload}: nbf {eng.nbf} (cart {eng.ncart}), ERI quartets {q_eri}, dERI quartets {q_deri}, "
        f"init {t_init:.2f} s; mixed @ {thr:g}: {n32 / max(n64 + n32, 1):.1%} of quartets in FP32")

    if args.copy_probe:
        src = torch.ones(64 << 20, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    # first-launch costs (code-object loading, side streams, the solver
    # libraries behind torch.linalg) stay out of the timings
    S0, T0, V0 = eng.oei()
    for prec in ((0,) if args.no_mixed else (0, 1)):
        eng.jk(S0, precision=prec, fp32_threshold=thr)
        eng.eri_grad(S0, precision=prec, fp32_threshold=thr)
    if not args.no_scf:
        from quax_amd.methods.hartree_fock import restricted_hartree_fock
        restricted_hartree_fock(eng, mol.nelectron(), {"diis": True, "spectral_shift": False, "maxit": 3})
    torch.cuda.synchronize()

    hf = {"fp32_threshold": thr, "fp32_quartet_fraction": n32 / max(n64 + n32, 1)}
    if args.no_scf:
        S, T, V = eng.oei()
        A = torch.linalg.inv(torch.linalg.cholesky(S)).T
        _, C2 = torch.linalg.eigh(A.T @ (T + V) @ A)
        Cocc = (A @ C2)[:, :mol.nelectron() // 2]
        D = (Cocc @ Cocc.T).contiguous()
    else:
        E, aux, grad, t_scf, t_grad = hf_energy_gradient(eng, mol, "fp64", thr)
        log(f"[bench] FP64 RHF E = {E:.10f} in {aux['iterations']} iterations ({t_scf:.2f} s), "
            f"gradient {t_grad:.3f} s, |sum g| = {abs(grad.reshape(-1, 3).sum(0)).max():.2e}")
        if args.no_mixed:
            raise SystemExit("--no-mixed needs --no-scf")
        Em, auxm, gradm, t_scfm, t_gradm = hf_energy_gradient(eng, mol, "mixed", thr)
        log(f"[bench] mixed RHF E = {Em:.10f} (error {Em - E:.2e}) in {auxm['iterations']} iterations "
            f"({t_scfm:.2f} s), gradient {t_gradm:.3f} s, max gradient error {np.abs(gradm - grad).max():.2e}")
        Eg, auxg, gradg, t_scfg, t_gradg = hf_energy_gradient(eng, mol, "fp64", thr, graph=True)
        log(f"[bench] graph-SCF RHF E = {Eg:.10f} (vs eager {Eg - E:.2e}) in {auxg['iterations']} iterations "
            f"({auxg.get('graph_iterations', auxg['iterations'])} replayed; {t_scfg:.2f} s), "
            f"max gradient difference {np.abs(gradg - grad).max():.2e}")
        hf.update({"scf_graph_wall_s": t_scfg, "scf_graph_iterations": auxg["iterations"],
                   "scf_graph_replays": auxg.get("graph_iterations", auxg["iterations"]),
                   "scf_graph_energy_vs_eager": Eg - E,
                   "scf_graph_grad_vs_eager": float(np.abs(gradg - grad).max())})
        D = aux["D"].contiguous()
        sweep = []
        for t in (float(x) for x in args.sweep.split(",") if x.strip()):
            n64t, n32t = eng.mixed_quartets(t)
            Et, auxt, gt, ts, tg = hf_energy_gradient(eng, mol, "mixed", t)
            sweep.append({"fp32_threshold": t, "fp32_quartet_fraction": n32t / max(n64t + n32t, 1),
                          "energy_error": Et - E, "grad_max_error": float(np.abs(gt - grad).max()),
                          "scf_iterations": auxt["iterations"], "wall_s": ts + tg})
            log(f"[bench] sweep {t:g}: FP32 {sweep[-1]['fp32_quartet_fraction']:.1%}, dE {Et - E:.2e}, "
                f"max dg {sweep[-1]['grad_max_error']:.2e}, {ts + tg:.2f} s")
        if sweep:
            hf["sweep"] = sweep
        hf.update({"energy": E, "scf_iterations": aux["iterations"], "scf_wall_s": t_scf, "grad_wall_s": t_grad,
                   "hf_gradient_wall_s_fp64": t_scf + t_grad,
                   "hf_gradient_wall_s_mixed": t_scfm + t_gradm, "scf_iterations_mixed": auxm["iterations"],
                   "energy_error_mixed": Em - E, "grad_max_error_mixed": float(np.abs(gradm - grad).max()),
                   "speedup_mixed": (t_scf + t_grad) / (t_scfm + t_gradm)})

    # headline: FP64 steps (J/K pass + adjoint gradient pass) on args.streams streams
    dt, _ = timed_steps(eng, D, args.steps, args.warmup, 0, 0.0, False)
    ms_step = dt * 1e3 / args.steps
    value = (q_eri + q_deri) / (dt / args.steps)
    dtm = None
    if not args.no_mixed:
        dtm, _ = timed_steps(eng, D, args.steps, 1, 1, thr, False)
    # roofline pass: the same steps on one stream, every kernel timed alone by
    # HIP events on its launch stream
    eng.set_streams(1)
    dts, (ms, launches, pq) = timed_steps(eng, D, args.steps, 0, 0, 0.0, True)
    eng.set_streams(args.streams)

    table = kernel_table(eng)
    eri_slots = [k for k in range(len(ms)) if table[k][3].startswith("jk")]
    eri_ms = float(ms[eri_slots].sum()) / args.steps
    deri_ms = float(ms.sum()) / args.steps - eri_ms
    slot = int(np.argmax(ms))
    name, fl = table[slot][:2]
    avg_ms = ms[slot] / launches[slot]
    model = flop_model()
    # roofline of the dominant kernel: ALGORITHMIC flops (textbook model) per launch
    alg_per_pq = slot_algorithmic_flops(table, model, eng, slot)
    flops_per_launch = alg_per_pq * pq[slot] / launches[slot]
    executed_per_launch = fl * pq[slot] / launches[slot]
    achieved = flops_per_launch / (avg_ms * 1e-3)
    total_flops = sum(table[k][1] * pq[k] for k in range(len(ms)) if launches[k]) / args.steps
    alg_step = sum(model["".join(map(str, l4))]["jk"] * ne + model["".join(map(str, l4))]["adjoint"] * nd
                   for (l4, ne, nd, _) in cq)
    kernels = sorted(((float(ms[k]) / args.steps, table[k][0], int(pq[k] // max(launches[k], 1)))
                      for k in range(len(ms)) if launches[k]), reverse=True)[:8]

    hf24 = None
    if args.workload == "cluster10" and not args.no_cluster24 and not args.no_mixed:
        # the metric's mixed-vs-FP64 HF-gradient wall time is quoted on the
        # 24-atom cluster (672 spherical functions)
        eng.close()
        hf24 = hf_mixed_vs_fp64(workloads.cluster24(), thr)
        eng = EriEngine(mol, basis, ints_tol=tol)

    cpu = None
    if args.cpu_seconds > 0:
        try:
            res, nthreads = cpu_baseline(mol, basis, tol, eng, args.cpu_seconds)
            r_e, n_e, t_e = res["eri"]
            r_d, n_d, t_d = res["deri"]
            t_cpu_step = q_eri / r_e + q_deri / r_d
            ncpu, cpu_model = host_cpu()
            cpu = {"value": (q_eri + q_deri) / t_cpu_step, "unit": "shell-quartets/s", "cores": nthreads,
                   "kind": "port", "host_logical_cpus": ncpu, "host_cpu_model": cpu_model,
                   "sample": f"{n_e} ERI + {n_d} dERI canonical screened quartets drawn uniformly from the same "
                             f"workload, CPU oracle (C, OpenMP {nthreads} threads; a clarity-first restatement "
                             f"that allocates per quartet, not Libint): ERI {r_e:.3g}/s, dERI "
                             f"{r_d:.3g}/s, combined over the step's mix"}
        except Exception as e:  # the baseline is reported, never required
            log(f"[bench] cpu baseline failed: {e}")

    out = {
        "metric": METRIC,
        "value": value,
        "unit": "shell-quartets/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": f"{args.workload}: {mol.natom()} atoms, {bname} "
                               f"{'spherical' if pure else 'Cartesian'} basis ({eng.nbf} AO / {eng.ncart} Cartesian), "
                               f"Schwarz 1e-12; step = direct J/K ERI pass + adjoint dERI gradient pass",
                   "eri_quartets": q_eri, "deri_quartets": q_deri, "streams": args.streams,
                   "one_stream_ms_per_step": dts * 1e3 / args.steps,
                   "eri_kernel_ms": eri_ms, "deri_kernel_ms": deri_ms},
        "roofline": {"bound": "valu", "bound_note": "FP64 vector ALU: the recurrences use no MFMA; MI355X FP64 "
                                                    "vector peak 78.6 TFLOP/s",
                     "achieved": achieved / 1e12, "peak": PEAK_FP64 / 1e12, "unit": "TFLOP/s",
                     "frac": achieved / PEAK_FP64, "traffic": measured_traffic(args.workload, name),
                     "traffic_unit": "bytes per launch (rocprofv3 FETCH_SIZE/WRITE_SIZE, copy-calibrated)",
                     "kernel": name, "avg_launch_ms": avg_ms,
                     "flops_per_launch": flops_per_launch, "flops_model": "quax_amd/csrc/flop_model.json",
                     "executed_flops_per_launch": executed_per_launch,
                     "step_algorithmic_flops": alg_step,
                     "step_algorithmic_tflops": alg_step / (ms_step * 1e-3) / 1e12,
                     "step_algorithmic_frac": alg_step / (ms_step * 1e-3) / PEAK_FP64,
                     "step_executed_flops": total_flops,
                     "step_executed_tflops": total_flops / (ms_step * 1e-3) / 1e12},
        "cpu_baseline": cpu,
        "mixed": None if dtm is None else
        {"fp32_threshold": thr, "ms_per_step": dtm * 1e3 / args.steps,
         "value": (q_eri + q_deri) / (dtm / args.steps), "speedup_vs_fp64_step": dt / dtm},
        "hf": hf,
        "hf_cluster24": hf24,
        "top_kernels_ms_per_step": kernels,
        "class_kernel_ms_per_step": class_times(table, ms, args.steps),
        "class_roofline": class_roofline(eng, model, class_times(table, ms, args.steps)),
    }
    print(json.dumps(out), flush=True)
    eng.close()


if __name__ == "__main__":
    main()
