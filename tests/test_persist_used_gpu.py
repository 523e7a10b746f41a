"""Which iterations run in one cooperative launch (clsparseAmdGetSolverLaunches), at
the sizes and diagonals where test_cg_persist_gpu.py and test_fsai_rows_gpu.py
compare them with separate launches; and the same comparison where the storage has
an even number of diagonals (the kernel of the next odd one reads 0 for the missing
diagonal) or one."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp
import torch

import clsparse_amd as cls
from clsparse_amd import fsai as fs
from gpu_helpers import cg_call, say
from test_cg_persist_gpu import CASES, _banded

pytestmark = pytest.mark.gpu


def _bicg(A, x, b, sc, ctl):
    lib = cls.load()
    fn = lib.clsparseScsrbicgStab if x.dtype == torch.float32 else lib.clsparseDcsrbicgStab
    xd, bd = cls.DenseVector(x), cls.DenseVector(b)
    return fn(ctypes.byref(xd.s), ctypes.byref(A.s), ctypes.byref(bd.s), sc.handle, ctl.handle)


def _solve(call, A, b, precond, iters, ctl, rel=1e-30):
    """x, iterations and (started, refused, gave up) of one solve from x = 0.25."""
    x = torch.full_like(b, 0.25)
    sc = cls.SolverControl(precond, iters, rel, 0.0)
    try:
        assert call(A, x, b, sc, ctl) == 0
        n = sc.launches()
        return x.cpu().numpy().astype(np.float64), sc.stats(), (n.started, n.refused, n.gave_up)
    finally:
        sc.release()


def _system(rp, ci, v, m, dtype, ctl):
    A = cls.CsrMatrix(rp, ci, v, m, dtype=dtype)
    A.meta_create(ctl)
    return A, torch.tensor(cls.gen_uniform(m, -1, 1, seed=m + 1).astype(dtype), device="cuda")


@pytest.mark.parametrize("n,offs,dtype,precond,sym", CASES,
                         ids=[f"{c[0]}-{len(c[1])}-{np.dtype(c[2]).name}-{'sym' if c[4] else 'full'}" for c in CASES])
def test_cg_runs_in_one_launch(monkeypatch, n, offs, dtype, precond, sym):
    say(f"cg launches n={n} offsets={offs}")
    with cls.Control() as ctl:
        A, b = _system(*_banded(n, offs, seed=n, sym=sym), dtype, ctl)
        assert _solve(cg_call, A, b, precond, 9, ctl)[2] == (1, 0, 0)
        monkeypatch.setenv("CLSPARSE_AMD_CG_PERSIST", "0")
        assert _solve(cg_call, A, b, precond, 9, ctl)[2] == (0, 0, 0)


@pytest.mark.parametrize("n,offs,dtype,sym", [
    (8, [1], np.float64, True), (513, [1], np.float64, False), (9393, [1, 93], np.float64, False),
    (70001, [1, 511, 512, 513], np.float32, False), (299993, [1, 100, 5000], np.float64, False),
    (299993, [1, 100, 5000], np.float64, True), (800000, [1, 110, 12345], np.float64, False),
    (1500000, [1, 110, 12345], np.float32, False)])
def test_bicgstab_runs_in_one_launch(n, offs, dtype, sym):
    say(f"bicgstab launches n={n} offsets={offs}")
    with cls.Control() as ctl:
        A, b = _system(*_banded(n, offs, seed=n + 5, sym=sym), dtype, ctl)
        for precond in (cls.DIAGONAL, cls.NOPRECOND):
            assert _solve(_bicg, A, b, precond, 5, ctl)[2] == (1, 0, 0)


@pytest.mark.parametrize("shape", [(12, 11, 10), (40, 37, 35), (100, 90, 110)])
@pytest.mark.parametrize("solver", ["mixed", "refined", "fsai"])
def test_refinement_solvers_run_in_one_launch(monkeypatch, solver, shape):
    say(f"{solver} launches {shape}")
    monkeypatch.setenv("CLSPARSE_AMD_FSAI_POLICY", "always")
    rp, ci, v, m = cls.gen_diffusion3d(*shape, sigma=1.0, ax=1.0, ay=1.0, az=10.0, seed=6)
    lib = cls.load()
    with cls.Control() as ctl:
        A, b = _system(rp, ci, v, m, np.float64, ctl)
        net = cls.Mlp(seed=1)
        net.set_params(fs.load_weights()[0])
        f = cls.Fsai(A, ctl)
        try:
            f.apply_net(net, ctl)

            def call(A, x, b, sc, ctl):
                xd, bd = cls.DenseVector(x), cls.DenseVector(b)
                args = (ctypes.byref(xd.s), ctypes.byref(A.s), ctypes.byref(bd.s))
                if solver == "fsai":
                    return lib.clsparseAmdDcsrcgFsai(*args, f.handle, sc.handle, ctl.handle)
                fn = lib.clsparseAmdDcsrcgMixed if solver == "mixed" else lib.clsparseAmdDcsrcgRefined
                return fn(*args, sc.handle, ctl.handle)

            _, stats, (started, refused, gave_up) = _solve(call, A, b, cls.DIAGONAL, 2000, ctl, rel=1e-9)
        finally:
            f.release()
            net.release()
    assert stats.status_detail == 0 and started >= 1 and refused == gave_up == 0


def test_systems_beyond_one_launch_use_none():
    say("solver launches: CSR matrix")
    rng = np.random.default_rng(4)
    a = sp.random(3000, 3000, density=4e-3, random_state=rng, format="csr")
    a = (a + a.T + sp.diags(np.full(3000, 20.0))).tocsr()
    a.sort_indices()
    with cls.Control() as ctl:
        A, b = _system(a.indptr.astype(np.uint32), a.indices.astype(np.uint32), a.data, 3000, np.float64, ctl)
        for call in (cg_call, _bicg):
            _, stats, n = _solve(call, A, b, cls.DIAGONAL, 200, ctl, rel=1e-8)
            assert n == (0, 0, 0) and stats.a_diagonals == 0 and stats.status_detail == 0


def _diagonals(n, offs, seed):
    """Diagonally dominant, nonzero on the given offsets only (0 among them)."""
    rng = np.random.default_rng(seed)
    diags = [np.full(n, 4.0 * len(offs)) + rng.uniform(0, 1, n) if k == 0 else -rng.uniform(0.2, 1.0, n - abs(k))
             for k in offs]
    a = sp.diags(diags, offs, shape=(n, n), format="csr")
    a.sort_indices()
    return a.indptr.astype(np.uint32), a.indices.astype(np.uint32), a.data, n


EVEN = [(600, [0, 1]), (513, [-1, 0]), (9393, [-93, -1, 0, 1]), (70001, [-5000, -3, 0, 2, 700, 701]),
        (299993, [-5000, -100, -1, 0, 1, 5000]), (400000, [-512, -511, -2, -1, 0, 1, 3, 513]),
        (800000, [-12345, -110, 0, 1, 110, 12345])]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,offs", EVEN + [(8, [0]), (700, [0]), (300000, [0])],
                         ids=[f"{n}-{len(o)}" for n, o in EVEN] + ["8-1", "700-1", "300000-1"])
def test_even_diagonal_counts_and_one(monkeypatch, n, offs, dtype):
    """Three iterations, as in test_cg_persist_gpu.py (1e-10 and 1e-5; BiCGStab
    1e-9 and 5e-5). A diagonal matrix with Jacobi is solved by the first one, so it
    runs without."""
    say(f"even diagonals n={n} offsets={offs} {np.dtype(dtype).name}")
    precond = cls.NOPRECOND if len(offs) == 1 else cls.DIAGONAL
    with cls.Control() as ctl:
        A, b = _system(*_diagonals(n, offs, seed=n), dtype, ctl)
        for call, tol in ((cg_call, 1e-10 if dtype == np.float64 else 1e-5),
                          (_bicg, 1e-9 if dtype == np.float64 else 5e-5)):
            monkeypatch.setenv("CLSPARSE_AMD_CG_PERSIST", "1")
            x1, s1, n1 = _solve(call, A, b, precond, 3, ctl)
            monkeypatch.setenv("CLSPARSE_AMD_CG_PERSIST", "0")
            x0, s0, n0 = _solve(call, A, b, precond, 3, ctl)
            assert n1 == (1, 0, 0) and n0 == (0, 0, 0)
            assert s1.a_diagonals == s0.a_diagonals == len(offs)
            assert s1.n_iters == s0.n_iters
            assert np.abs(x1 - x0).max() <= tol * np.abs(x0).max()


@pytest.mark.parametrize("solver", ["cg", "bicgstab", "mixed"])
def test_give_ups_are_counted(monkeypatch, solver):
    say(f"give-ups of {solver}")
    monkeypatch.setenv("CLSPARSE_AMD_PERSIST_SPIN", "1")
    rp, ci, v, m = cls.gen_diffusion3d(40, 37, 35, sigma=1.0, ax=1.0, ay=1.0, az=10.0, seed=6)
    lib = cls.load()

    def mixed(A, x, b, sc, ctl):
        xd, bd = cls.DenseVector(x), cls.DenseVector(b)
        return lib.clsparseAmdDcsrcgMixed(ctypes.byref(xd.s), ctypes.byref(A.s), ctypes.byref(bd.s), sc.handle,
                                          ctl.handle)

    with cls.Control() as ctl:
        A, b = _system(rp, ci, v, m, np.float64, ctl)
        call = {"cg": cg_call, "bicgstab": _bicg, "mixed": mixed}[solver]
        _, stats, n = _solve(call, A, b, cls.DIAGONAL, 5000, ctl, rel=1e-9)
    assert n == (1, 0, 1) and stats.status_detail == 0
