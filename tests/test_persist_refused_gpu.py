"""A cooperative launch that the device refuses (CLSPARSE_AMD_PERSIST_REFUSE=1: taken
as refused) has run nothing: the solve goes on as if there were no such launches, with
the same bits as with CLSPARSE_AMD_CG_PERSIST=0. The control's host buffer then holds
what an earlier solve left there; here one of another kind, whose words at the place
of the new solve's are not 0."""
import ctypes

import numpy as np
import pytest
import torch

import clsparse_amd as cls
from gpu_helpers import cg_call, say

pytestmark = pytest.mark.gpu


def _call(name):
    if name == "cg":
        return cg_call
    fn = {"bicgstab": "clsparseDcsrbicgStab", "mixed": "clsparseAmdDcsrcgMixed", "refined": "clsparseAmdDcsrcgRefined"}

    def call(A, x, b, sc, ctl):
        xd, bd = cls.DenseVector(x), cls.DenseVector(b)
        return getattr(cls.load(), fn[name])(ctypes.byref(xd.s), ctypes.byref(A.s), ctypes.byref(bd.s), sc.handle,
                                             ctl.handle)
    return call


@pytest.mark.parametrize("first,solver", [("bicgstab", "cg"), ("bicgstab", "mixed"), ("bicgstab", "refined"),
                                          ("cg", "bicgstab")])
def test_refused_launch_runs_as_without(monkeypatch, first, solver):
    say(f"refused launches of {solver} after {first}")
    rp, ci, v, m = cls.gen_poisson2d(60, 50)
    b = torch.tensor(cls.gen_uniform(m, -1, 1, seed=3), device="cuda")
    out = {}
    for env in ("CLSPARSE_AMD_CG_PERSIST", "CLSPARSE_AMD_PERSIST_REFUSE"):
        with cls.Control() as ctl:
            A = cls.CsrMatrix(rp, ci, v, m)
            A.meta_create(ctl)
            sc = cls.SolverControl(cls.DIAGONAL, 500, 1e-9, 0.0)
            assert _call(first)(A, torch.zeros_like(b), b, sc, ctl) == 0
            assert sc.launches().started == 1
            sc.release()
            monkeypatch.setenv(env, "0" if env.endswith("PERSIST") else "1")
            # The initial residual counts: 1 / 1000 of it ends CG and BiCGStab.
            sc = cls.SolverControl(cls.DIAGONAL, 500, 1e-9 if solver in ("mixed", "refined") else 0.0, 1e-3)
            x = torch.full_like(b, 0.25)
            assert _call(solver)(A, x, b, sc, ctl) == 0
            n, st = sc.launches(), sc.stats()
            sc.release()
            monkeypatch.delenv(env)
            assert (n.started, n.refused, n.gave_up) == (0, 0 if env.endswith("PERSIST") else 1, 0)
            assert st.status_detail == 0
            out[env] = (x.cpu().numpy(), st.n_iters, st.outer_iterations, st.initial_residual)
    a, r = out.values()
    assert a[1:] == r[1:]
    np.testing.assert_array_equal(a[0], r[0])
