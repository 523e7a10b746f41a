"""A launch that gives up in the pilot race of a learned solve, whose two engines share
the slots of the grid-wide sums: neither starts another one, and the solve reaches its
tolerance (true residual)."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp
import torch

import clsparse_amd as cls
from clsparse_amd import fsai as fs
from gpu_helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", ["trained", "random"])
def test_neither_engine_launches_again(monkeypatch, weights):
    say(f"give-up in the pilot race, {weights} network")
    monkeypatch.setenv("CLSPARSE_AMD_PERSIST_SPIN", "1")
    monkeypatch.setenv("CLSPARSE_AMD_FSAI_POLICY", "race")
    rp, ci, v, m = cls.gen_diffusion3d(40, 37, 35, sigma=1.0, ax=1.0, ay=1.0, az=100.0, seed=6)
    b = cls.gen_uniform(m, -1, 1, seed=3)
    with cls.Control() as ctl:
        A = cls.CsrMatrix(rp, ci, v, m)
        A.meta_create(ctl)
        net = cls.Mlp(seed=1)
        if weights == "trained":
            net.set_params(fs.load_weights()[0])
        f = cls.Fsai(A, ctl)
        f.apply_net(net, ctl)
        sc = cls.SolverControl(cls.DIAGONAL, 5000, 1e-9, 0.0)
        x = torch.zeros(m, dtype=torch.float64, device="cuda")
        xd, bd = cls.DenseVector(x), cls.DenseVector(torch.tensor(b, device="cuda"))
        try:
            assert cls.load().clsparseAmdDcsrcgFsai(ctypes.byref(xd.s), ctypes.byref(A.s), ctypes.byref(bd.s), f.handle,
                                                    sc.handle, ctl.handle) == 0
            n, st = sc.launches(), sc.stats()
        finally:
            sc.release()
            f.release()
            net.release()
    assert st.pilot_rate_fsai != 0 and st.pilot_rate_jacobi != 0  # both engines ran
    assert (n.started, n.refused, n.gave_up) == (1, 0, 1)
    a = sp.csr_matrix((v, ci, rp), shape=(m, m))
    assert np.linalg.norm(b - a @ x.cpu().numpy()) <= 1.01e-9 * np.linalg.norm(b)
