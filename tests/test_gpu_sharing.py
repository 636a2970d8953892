"""Passes that share a context, a stream or a capture with others.

Results are compared with the same entry point called alone: FP64 sums of the
same terms, whose order differs by atomics only, so 1e-12 of the largest
element."""
import ctypes

import numpy as np
import pytest

from quax_amd.basis import BasisSet
from quax_amd.molecule import synthetic_cluster

pytestmark = pytest.mark.gpu


def _density(n, seed):
    X = np.random.default_rng(seed).standard_normal((n, n)) * 0.3
    return X @ X.T / n


def _same(a, b):
    assert bool(a.isfinite().all())
    assert (a - b).abs().max().item() <= 1e-12 * max(1.0, b.abs().max().item())


def _noalloc(eng, D, J, K):
    from quax_amd import _lib
    _lib.check(eng.L.qx_jk_build_noalloc(eng.ctx, _lib.ptr(D), _lib.ptr(J), _lib.ptr(K), eng._stream()), eng.ctx)


def _context(basis, pure):
    from quax_amd.engine import EriEngine
    mol = synthetic_cluster(2, 1, 11, n_o=1) if basis == "sto-3g" else synthetic_cluster(3, 1, 11)
    return EriEngine(mol, BasisSet.build(mol, basis, pure=pure), ints_tol=1e-12)


@pytest.mark.parametrize("basis,pure", [("sto-3g", False), ("even-tempered", True)])
def test_noalloc_pass_beside_another_pass(gpu, basis, pure):
    """Both passes in flight on two streams of one context, with densities of
    different size, and a captured allocation-free pass replayed beside the other."""
    torch = gpu
    with _context(basis, pure) as eng:
        n = eng.nbf
        D1, D2 = (torch.as_tensor(_density(n, k) * s, device="cuda") for k, s in ((1, 1.0), (2, 50.0)))
        ref1, ref2 = [x.clone() for x in eng.jk(D1)], [x.clone() for x in eng.jk(D2)]
        new = lambda: torch.full((n, n), float("nan"), dtype=torch.float64, device="cuda")
        J, K, Jg, Kg = new(), new(), new(), new()
        s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            _noalloc(eng, D1, Jg, Kg)
        for rep in range(12):
            out = (new(), new())
            torch.cuda.synchronize()
            with torch.cuda.stream(s1):
                if rep % 2:
                    graph.replay()
                else:
                    _noalloc(eng, D1, J, K)
            with torch.cuda.stream(s2):
                eng.jk(D2, out=out)
            torch.cuda.synchronize()
            for got, want in zip((Jg, Kg) if rep % 2 else (J, K), ref1):
                _same(got, want)
            for got, want in zip(out, ref2):
                _same(got, want)


@pytest.mark.parametrize("basis,pure", [("sto-3g", False), ("even-tempered", True)])
def test_noalloc_pass_uses_no_events(gpu, basis, pure):
    torch = gpu
    with _context(basis, pure) as eng:
        n = eng.nbf
        D = torch.as_tensor(_density(n, 3), device="cuda")
        J, K = (torch.empty((n, n), dtype=torch.float64, device="cuda") for _ in range(2))
        eng.profile(True)
        _noalloc(eng, D, J, K)
        assert eng.profile_read()[1].sum() == 0
        for got, want in zip((J, K), eng.jk(D)):
            _same(got, want)
        assert eng.profile_read()[1].sum() > 0


@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("basis,pure", [("sto-3g", False), ("even-tempered", False), ("even-tempered", True)])
def test_captured_tensor_passes(gpu, basis, pure, warm):
    """Integral and first-derivative tensors under capture, in a fresh context and
    in one whose workspace other passes have used, replayed between eager passes
    that use and give back that workspace."""
    torch = gpu
    from quax_amd.engine import EriEngine
    mol = synthetic_cluster(1, 1, 5)
    calls = [lambda e: e.compute_2e_int(), lambda e: e.eri_deriv_core(1),
             lambda e: e.compute_2e_deriv([0] * 6), lambda e: e.compute_2e_deriv([0, 0, 0, 0, 1, 0])]
    with EriEngine(mol, BasisSet.build(mol, basis, pure=pure), ints_tol=1e-12) as ref_eng:
        ref = [f(ref_eng).clone() for f in calls]
    for f, want in zip(calls, ref):
        with EriEngine(mol, BasisSet.build(mol, basis, pure=pure), ints_tol=1e-12) as eng:
            D = torch.as_tensor(_density(eng.nbf, 4), device="cuda")
            if warm:
                calls[1](eng)
                eng.jk(D)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = f(eng)
            for rep in range(4):
                out.fill_(float("nan"))
                graph.replay()
                torch.cuda.synchronize()
                _same(out, want)
                for other, w in zip(calls, ref):
                    _same(other(eng), w)
                eng.jk(D)
                if rep == 1:
                    eng.set_tensor_limit(1 << 30)
                    eng.set_tensor_limit(0)


def _kernels(torch, call):
    """Kernel launches of a call, from the graph it is captured into."""
    hip = ctypes.CDLL("libamdhip64.so")
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    raw, n = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    kinds = [ctypes.c_int() for _ in nodes]
    assert all(hip.hipGraphNodeGetType(ctypes.c_void_p(x), ctypes.byref(k)) == 0 for x, k in zip(nodes, kinds))
    return sum(k.value == 0 for k in kinds)


@pytest.mark.parametrize("setter,value,pass_", [("set_class_tiles", 192, 0), ("set_jk_rows", 0, 0),
                                                ("set_class_tiles", 192, 1), ("set_grad_copies", 2, 1),
                                                ("set_grad_wave_reduce", None, 1)])
def test_tuning_calls_reach_small_molecules(gpu, setter, value, pass_):
    """A small s, p molecule's one launch gives way to the class kernels that a
    tuning call addresses, with the same results, and comes back with the defaults."""
    torch = gpu
    with _context("sto-3g", False) as eng:
        D = torch.as_tensor(_density(eng.nbf, 5), device="cuda")
        out = [torch.empty((eng.nbf, eng.nbf), dtype=torch.float64, device="cuda") for _ in range(2)]
        run = (lambda: eng.jk(D, out=out)) if pass_ == 0 else (lambda: (eng.eri_grad(D),))
        want = [x.clone() for x in run()]
        one = _kernels(torch, run)
        set_ = getattr(eng, setter)
        args = (pass_,) if setter == "set_class_tiles" else ()
        n = len(eng.jk_rows())
        flags = [value] * n if value is not None else [not f for f in eng.grad_wave_reduce()]
        set_(*args, flags)
        for got, w in zip(run(), want):
            _same(got, w)
        assert _kernels(torch, run) >= one + 5  # six class lists at least
        set_(*args, None)
        assert _kernels(torch, run) == one
        for got, w in zip(run(), want):
            _same(got, w)


def test_captured_tensor_pass_in_slices(gpu):
    torch = gpu
    from quax_amd.engine import EriEngine
    mol = synthetic_cluster(1, 1, 5)
    with EriEngine(mol, BasisSet.build(mol, "sto-3g", pure=False), ints_tol=1e-12) as eng:
        want = eng.eri_deriv_core(1).clone()
        for limit in (24 * 24 * 8 * 2, 4096):  # two of six slices; row panels
            eng.set_tensor_limit(limit)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = eng.eri_deriv_core(1)
            for _ in range(3):
                out.fill_(float("nan"))
                graph.replay()
                torch.cuda.synchronize()
                _same(out, want)
                _same(eng.eri_deriv_core(1), want)
