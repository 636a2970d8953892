"""Each choice between kernels at the sizes where it can go wrong, against the
other path, the oracle or an independent algorithm.

Tolerances: every comparison is between FP64 sums of the same terms in another
order.  With elements below 1e2 and some 1e4 terms per element the difference
is of the order of 1e2 * eps * sqrt(1e4) = 2e-12 in the worst element and far
less in most; 1e-11 absolute is used (times the largest element where that
exceeds 1e2)."""
import numpy as np
import pytest

import oracle
from quax_amd.basis import BasisSet, Shell
from quax_amd.molecule import Molecule, synthetic_cluster

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _density(n, seed):
    X = np.random.default_rng(seed).standard_normal((n, n)) * 0.3
    return X @ X.T / np.sqrt(n)


def _engine(mol, bs, **kw):
    from quax_amd.engine import EriEngine
    return EriEngine(mol, bs, **kw)


def _close(a, b, tol=TOL):
    a, b = (x.cpu().numpy() if hasattr(x, "cpu") else np.asarray(x) for x in (a, b))
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= tol * max(1.0, np.abs(b).max() / 1e2)


def _shells(atoms, spec):
    """spec: per shell (l, exponents); unit coefficients, on every atom."""
    return [Shell(l, a, list(e), [1.0] * len(e)) for a in range(atoms) for l, e in spec]


def _line(n, dist):
    return Molecule(["C"] * n, np.array([[0.0, 0.1 * k, dist * k] for k in range(n)]))


@pytest.mark.parametrize("symbols", [["H"], ["H", "H"], ["O", "H", "H"], ["C"] * 5 + ["H"] * 5, ["C"] * 7 + ["H"] * 6])
def test_one_launch_pass_equals_separate_kernels(gpu, symbols):
    """s and p molecules from one function to both sides of the size limit;
    profiled passes run the class kernels one by one."""
    n_c, n_o, n_h = (symbols.count(x) for x in "COH")
    mol = synthetic_cluster(n_c, n_h, 3, n_o=n_o) if len(symbols) > 1 else Molecule(symbols, np.zeros((1, 3)))
    bs = BasisSet.build(mol, "sto-3g", pure=False)
    D = _density(bs.nbf(), 1)
    with _engine(mol, bs, ints_tol=1e-12) as eng:
        one = (*eng.jk(D), eng.eri_grad(D))
        eng.profile(True)
        for a, b in zip(one, (*eng.jk(D), eng.eri_grad(D))):
            _close(a, b)


@pytest.mark.parametrize("prims", [1, 2, 7])
@pytest.mark.parametrize("dist", [0.9, 3.0, 40.0])
def test_quadrature_tensor_against_hermite_j_and_k(gpu, dist, prims):
    """The tensor of s, p, d shells (quadrature for the heavy classes, arguments
    from 0 to beyond the root tables) contracted to J and K, against the J
    engine and the K kernels."""
    import torch
    exps = np.geomspace(9.0, 0.4, prims) if prims > 1 else np.array([0.8])
    mol = _line(2, dist)
    bs = BasisSet("mixed", _shells(2, [(0, exps), (1, exps), (2, exps), (2, [1.7])]), pure=False)
    D = _density(bs.nbf(), 2)
    with _engine(mol, bs, ints_tol=1e-14) as eng:
        G, Dt = eng.compute_2e_int(), torch.as_tensor(D, device="cuda")
        n = eng.nbf
        J, K = eng.jk(D)
        _close(J, (G.reshape(n * n, n * n) @ Dt.reshape(-1)).reshape(n, n))
        _close(K, (G.permute(0, 2, 1, 3).reshape(n * n, n * n) @ Dt.reshape(-1)).reshape(n, n))


@pytest.mark.parametrize("pure", [False, True])
@pytest.mark.parametrize("slices", [1, 4])
def test_tensors_in_slices_equal_whole(gpu, pure, slices):
    mol = _line(3, 2.1)
    bs = BasisSet("spd", _shells(3, [(0, [0.9]), (1, [1.1]), (2, [0.7])]), pure=pure)
    with _engine(mol, bs, ints_tol=1e-14) as eng:
        whole = eng.eri_deriv_core(1)
        ld = (sum(len(_comp(a)) * len(_comp(b)) for a, b in _pairs(bs)) + 7) // 8 * 8
        eng.set_tensor_limit(slices * ld * ld * 8)
        _close(eng.eri_deriv_core(1), whole)


def _comp(l):
    return range((l + 1) * (l + 2) // 2)


def _pairs(bs):
    ls = [s.l for s in bs.shells]
    return [(ls[i], ls[j]) for i in range(len(ls)) for j in range(i + 1)]


def test_tensors_in_row_panels_equal_whole(gpu):
    """Less than one slice: panels of rows, scattered (Cartesian; a spherical
    tensor needs its slice)."""
    from quax_amd._lib import QuaxNativeError
    mol = _line(3, 2.1)
    spec = [(0, [0.9]), (1, [1.1]), (2, [0.7])]
    for pure in (False, True):
        bs = BasisSet("spd", _shells(3, spec), pure=pure)
        with _engine(mol, bs, ints_tol=1e-14) as eng:
            whole, deriv = eng.compute_2e_int(), eng.eri_deriv_core(1)
            eng.set_tensor_limit(4096)
            if pure:
                with pytest.raises(QuaxNativeError):
                    eng.compute_2e_int()
                eng.set_tensor_limit(0)
            _close(eng.compute_2e_int(), whole)
            _close(eng.eri_deriv_core(1), deriv)


def _three_atoms(kind, pure):
    from quax_amd.engine import EriEngine
    mol = _line(3, 2.1)
    more = [2.5, 0.8] if kind == "contracted" else []
    bs = BasisSet("spd", _shells(3, [(0, [0.9] + more), (1, [1.1] + more), (2, [0.7])]), pure=pure)
    return EriEngine(mol, bs, ints_tol=1e-14, fragments=[0, 1, 0] if kind == "fragments" else None)


@pytest.mark.parametrize("kind", ["single", "contracted", "fragments"])
def test_tensors_in_many_row_panels(gpu, kind):
    """36 rows at a time: every dd pair is a panel of its own, in one slice per
    pass, so panels and slices start inside their lists."""
    import ctypes
    with _three_atoms(kind, False) as eng:
        whole = eng.compute_2e_int(), eng.eri_deriv_core(1), eng.eri_deriv_core(2)
        eng.set_tensor_limit(4096)
        eng.profile(True)
        panels = eng.compute_2e_int()
        launches = eng.profile_read()[1]
        eng.profile(False)
        l4, most = (ctypes.c_int * 4)(), {}
        for slot in np.flatnonzero(launches):
            k, c, p, f = (ctypes.c_int() for _ in range(4))
            eng.L.qx_profile_slot(int(slot), *(ctypes.byref(x) for x in (k, c, p, f)))
            eng.L.qx_class_info(c.value, l4, None)
            most[tuple(l4)] = launches[slot]
        assert most[2, 2, 2, 2] == (4 if kind == "fragments" else 6) and most[2, 1, 0, 0] > 1
        _close(panels, whole[0])
        _close(eng.eri_deriv_core(1), whole[1])
        _close(eng.eri_deriv_core(2), whole[2])


@pytest.mark.parametrize("pure", [False, True])
def test_second_derivative_tensor_in_slices(gpu, pure):
    with _three_atoms("contracted", pure) as eng:
        whole = eng.eri_deriv_core(2)
        eng.set_tensor_limit(4 * 520 * 520 * 8)  # four of nine slices
        _close(eng.eri_deriv_core(2), whole)
        _close(eng.compute_2e_deriv([1, 0, 0, 0, 0, 0, 0, 0, 1]), whole[8])


def test_kept_tensor_workspace_is_given_back(gpu):
    torch = gpu
    mol = _line(2, 2.1)
    bs = BasisSet("spd", _shells(2, [(0, [0.9]), (1, [1.1]), (2, [0.7]), (2, [1.9]), (2, [0.3])]), pure=True)
    with _engine(mol, bs, ints_tol=1e-14) as eng:
        eng.set_tensor_limit(0)
        free = lambda: torch.cuda.mem_get_info()[0]
        out = eng.eri_deriv_core(1)
        held = free()
        eng.set_tensor_limit(10 * 1024 * 1024)  # one slice
        assert free() > held
        _close(eng.eri_deriv_core(1), out)


@pytest.mark.parametrize("n_c,pure", [(1, True), (2, False), (7, True)])
def test_expansion_of_a_tensor(gpu, n_c, pure):
    """28 functions of one carbon (one workgroup's triangle, even rows), 60
    Cartesian ones, and 196, beyond the largest triangle: J from the tensor."""
    import torch
    mol = synthetic_cluster(n_c, 0, 9) if n_c > 1 else Molecule(["C"], np.zeros((1, 3)))
    bs = BasisSet.build(mol, "even-tempered", pure=pure)
    D = _density(bs.nbf(), 4)
    with _engine(mol, bs, ints_tol=1e-12) as eng:
        n = eng.nbf
        G = eng.compute_2e_int()
        J = (G.reshape(n * n, n * n) @ torch.as_tensor(D, device="cuda").reshape(-1)).reshape(n, n)
        _close(eng.jk(D)[0], J)
        if n > 100:  # symmetric under exchange of the pairs and within each
            assert torch.equal(G[3, 7], G[7, 3])
            _close(G[3, 7], G[:, :, 3, 7])


@pytest.mark.parametrize("rows", [0, 1])
def test_k_rows_in_lds_or_not(gpu, rows):
    """K' in LDS rows or by global atomics, for every class."""
    mol = _line(2, 2.3)
    bs = BasisSet("spd", _shells(2, [(0, [0.9]), (1, [1.1]), (2, [0.7]), (2, [2.0, 0.3])]), pure=False)
    D = _density(bs.nbf(), 5)
    ob = oracle.OracleBasis(mol, bs)
    G = ob.compute_2e_int(1e-14)
    with _engine(mol, bs, ints_tol=1e-14) as eng:
        eng.set_jk_rows([rows] * len(eng.jk_rows()))
        J, K = eng.jk(D)
    _close(J, np.einsum("pqrs,rs->pq", G, D))
    _close(K, np.einsum("prqs,rs->pq", G, D))


@pytest.mark.parametrize("case", ["spherical", "cartesian", "many atoms"])
def test_one_electron_gradient_against_derivative_matrices(gpu, case):
    """The contracted kernels (nuclei shared by eight lanes) against the
    derivative matrices' kernel; 260 atoms are beyond the LDS accumulators."""
    import torch
    if case == "many atoms":
        grid = np.array([[x, y, z] for x in range(7) for y in range(7) for z in range(6)], float)[:260] * 2.0
        mol = Molecule(["H"] * 260, grid)
        bs = BasisSet("s", _shells(260, [(0, [0.8])]), pure=False)
    else:
        mol = _line(3, 2.0)
        bs = BasisSet("spd", _shells(3, [(0, [3.0, 0.5]), (1, [1.1]), (2, [0.7])]), pure=case == "spherical")
    P, W = _density(bs.nbf(), 6), _density(bs.nbf(), 7)
    with _engine(mol, bs, ints_tol=1e-12) as eng:
        g = eng.oei_grad(P, W)
        dS, dT, dV = eng.oei_deriv()
        Pt, Wt = (torch.as_tensor(x, device="cuda") for x in (P, W))
        _close(g.reshape(-1), ((dT + dV) * Pt).sum((1, 2)) + (dS * Wt).sum((1, 2)))


@pytest.mark.parametrize("n,m", [((4, 3, 5, 6), (129, 16, 17, 1)), ((4, 3, 5, 6), (128, 112, 15, 113)),
                                 ((41, 40, 40, 3), (2, 3, 2, 17))])
def test_transformation_tile_edges(gpu, n, m):
    """Row tiles of 16 and panels of 128, and the wide column tiles."""
    from quax_amd.methods.energy_utils import partial_tei_transformation
    rng = np.random.default_rng(8)
    G = rng.standard_normal(n)
    C = [rng.standard_normal((n[k], m[k])) for k in range(4)]
    ref = G
    for c in C:
        ref = np.tensordot(ref, c, axes=[(0,), (0,)])
    _close(partial_tei_transformation(G, *C), ref)


@pytest.mark.parametrize("prims", [1, 3])
@pytest.mark.parametrize("pure", [False, True])
def test_directional_jk_against_the_derivative_tensor(gpu, pure, prims):
    """The dual-number J and K kernels of every class against the first-derivative
    tensor contracted with the direction and the density."""
    import torch
    mol = Molecule(["C", "O", "C"], np.array([[0.0, 0.1, -0.3], [1.3, 2.0, 0.4], [-1.1, 0.9, 2.2]]))
    geo = lambda x: list(x * 2.5 ** np.arange(prims))
    bs = BasisSet("spd", _shells(3, [(0, geo(0.5)), (1, geo(0.4)), (2, geo(0.6))]), pure=pure)
    D = _density(bs.nbf(), 10)
    v = np.random.default_rng(11).standard_normal(9)
    with _engine(mol, bs, ints_tol=1e-14) as eng:
        n = eng.nbf
        G = torch.tensordot(torch.as_tensor(v, device="cuda"), eng.eri_deriv_core(1), dims=1)
        J, K = eng.jk_deriv_dir(D, v)
        Dt = torch.as_tensor(D, device="cuda").reshape(-1)
        _close(J, (G.reshape(n * n, n * n) @ Dt).reshape(n, n))
        _close(K, (G.permute(0, 2, 1, 3).reshape(n * n, n * n) @ Dt).reshape(n, n))


def _molecules_as_fragments():
    """Uneven molecules of s and p shells side by side, and each by itself."""
    mols = [synthetic_cluster(0, 2, 3, n_o=1), synthetic_cluster(2, 1, 4), Molecule(["H"], np.zeros((1, 3))),
            synthetic_cluster(1, 4, 6)]
    xyz = np.vstack([np.asarray(m.geometry()).reshape(-1, 3) + [0.0, 0.0, 25.0 * k] for k, m in enumerate(mols)])
    sym = [m.symbol(i) for m in mols for i in range(m.natom())]
    frag = [k for k, m in enumerate(mols) for _ in range(m.natom())]
    return mols, Molecule(sym, xyz), frag


def test_one_launch_passes_and_tensors_of_fragments(gpu):
    """The one-launch J/K (whole and with fragments left out), the gradient and the
    tensors of a batch of minimal-basis molecules against one context each."""
    import torch
    mols, comb, frag = _molecules_as_fragments()
    nb = [BasisSet.build(m, "sto-3g").nbf() for m in mols]
    off = np.concatenate([[0], np.cumsum(nb)])
    D = np.zeros((off[-1],) * 2)
    for k, n in enumerate(nb):
        D[off[k]:off[k + 1], off[k]:off[k + 1]] = _density(n, 20 + k)
    with _engine(comb, BasisSet.build(comb, "sto-3g"), ints_tol=1e-14, fragments=frag) as eng:
        J, K = eng.jk(D)
        skip = [0, 1, 0, 1]
        Js, Ks = eng.jk(D, frag_skip=skip)
        g = eng.eri_grad(D).reshape(-1, 3)
        G, dG = eng.compute_2e_int(), eng.eri_deriv_core(1)
    inside = torch.zeros_like(G, dtype=torch.bool)
    at = 0
    for k, m in enumerate(mols):
        s = slice(off[k], off[k + 1])
        a = slice(at, at + m.natom())
        at += m.natom()
        inside[s, s, s, s] = True
        with _engine(m, BasisSet.build(m, "sto-3g"), ints_tol=1e-14) as one:
            Jk, Kk = one.jk(D[s, s])
            _close(J[s, s], Jk)
            _close(K[s, s], Kk)
            _close(Js[s, s], Jk * (1 - skip[k]))
            _close(Ks[s, s], Kk * (1 - skip[k]))
            _close(g[a], one.eri_grad(D[s, s]).reshape(-1, 3))
            _close(G[s, s, s, s], one.compute_2e_int())
            _close(dG[3 * a.start:3 * a.stop, s, s, s, s], one.eri_deriv_core(1))
    assert (G[~inside] == 0).all() and (dG[:, ~inside] == 0).all()


@pytest.mark.parametrize("n_c,extra,offset", [(1, 0, 1), (2, 1, 0), (2, 1, 1), (7, 1, 0), (7, 2, 1)])
def test_expansion_odd_or_unaligned(gpu, n_c, extra, offset):
    """An odd number of functions, and an output off its 16-byte line, on both
    sides of the largest triangle: no wide stores."""
    import torch
    from quax_amd import _lib
    mol = synthetic_cluster(n_c, 0, 9) if n_c > 1 else Molecule(["C"], np.zeros((1, 3)))
    bs = BasisSet.build(mol, "even-tempered", pure=True)
    bs = BasisSet("more", bs.shells + [Shell(0, 0, [0.05 * 3 ** k], [1.0]) for k in range(extra)], pure=True)
    with _engine(mol, bs, ints_tol=1e-12) as eng:
        n = eng.nbf
        assert n % 2 == extra % 2 and (n > 195) == (n_c == 7)
        buf = torch.full((n ** 4 + 2,), float("nan"), dtype=torch.float64, device="cuda")
        out = buf[offset:offset + n ** 4]
        assert out.data_ptr() % 16 == 8 * offset
        _lib.check(eng.L.qx_compute_2e_int(eng.ctx, _lib.ptr(out), eng._stream()), eng.ctx)
        assert torch.isnan(buf[:offset]).all() and torch.isnan(buf[offset + n ** 4:]).all()
        D = _density(n, 21)
        J = (out.view(n * n, n * n) @ torch.as_tensor(D, device="cuda").reshape(-1)).reshape(n, n)
        _close(eng.jk(D)[0], J)
