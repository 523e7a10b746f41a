"""csrmm on rows far longer than the mean, which all slots of a wave share (more than 16
trips of a slot and eight times the mean), next to those that the workgroup takes
(more than 512 entries), for every slot width; and products with few rows, which
take one column per lane where 16 bytes of columns do not divide their count.

Tolerance as in test_csrmm_rows_gpu.py; two calls give the same bits."""
import ctypes

import numpy as np
import pytest
import torch

import clsparse_amd as cls
import oracle
from gpu_helpers import random_csr, say
from test_csrmm_gpu import _dense

pytestmark = pytest.mark.gpu


def _check(lens, m, ncols, dtype, alpha, beta):
    rng = np.random.default_rng(ncols)
    rp, ci, v = random_csr(rng, lens, m)
    v = v.astype(dtype)
    n = rp.size - 1
    B = rng.uniform(-1, 1, (m, ncols + 2)).astype(dtype)
    C0 = rng.uniform(-1, 1, (n, ncols + 1)).astype(dtype)
    if beta == 0:
        C0[:, :ncols] = np.nan
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    fn = cls.load().clsparseScsrmm if dtype == np.float32 else cls.load().clsparseDcsrmm
    got = []
    with cls.Control() as ctl:
        A = cls.CsrMatrix(rp, ci, v, m, dtype=dtype)
        a, b = cls.Scalar(alpha, tdt), cls.Scalar(beta, tdt)
        Bt = torch.tensor(B.ravel(), device="cuda")
        for _ in range(2):
            Ct = torch.tensor(C0.ravel(), device="cuda")
            Bd, Cd = _dense(Bt, m, ncols, ncols + 2), _dense(Ct, n, ncols, ncols + 1)
            cls.check("csrmm", fn(ctypes.byref(a.s), ctypes.byref(A.s), ctypes.byref(Bd), ctypes.byref(b.s),
                                  ctypes.byref(Cd), ctl.handle))
            got.append(Ct.cpu().numpy().reshape(n, ncols + 1))
    np.testing.assert_array_equal(got[0], got[1])
    np.testing.assert_array_equal(got[0][:, ncols], C0[:, ncols])  # padding untouched
    ref, scale = oracle.csrmm(rp, ci, v.astype(np.float64), B[:, :ncols].astype(np.float64),
                              np.where(np.isnan(C0), 0, C0)[:, :ncols].astype(np.float64), alpha, beta)
    bound = np.maximum(1e-6 if dtype == np.float32 else 1e-13, (lens + 4) * np.finfo(dtype).eps)[:, None]
    assert np.all(np.abs(got[0][:, :ncols].astype(np.float64) - ref) <= bound * scale)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("alpha,beta", [(-0.75, 0.5), (1.0, 0.0), (0.0, 2.0)])
@pytest.mark.parametrize("ncols", [1, 2, 3, 4, 5, 8, 13, 20, 33, 64, 70])
def test_rows_far_longer_than_the_mean(ncols, alpha, beta, dtype):
    say(f"csrmm far rows ncols={ncols} alpha={alpha} {np.dtype(dtype).name}")
    rng = np.random.default_rng(3)
    lens = rng.integers(0, 7, 40_000)
    # On both sides of 16 trips of every slot width (16 W entries), several to a wave.
    edge = np.concatenate([[16 * w + d for w in (1, 2, 4, 8, 16, 32) for d in (-1, 0, 1, 7)], [511, 512, 513, 900]])
    lens[rng.choice(lens.size, 5 * edge.size, replace=False)] = np.tile(edge, 5)
    lens[800:840] = 300
    lens[-1] = 200
    _check(lens, 3000, ncols, dtype, alpha, beta)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ncols", [1, 3, 5, 6, 7, 9, 13, 17, 31, 33, 63, 65, 130])
@pytest.mark.parametrize("n,mean", [(1, 40), (37, 9), (500, 81), (1850, 4)])
def test_few_rows(n, mean, ncols, dtype):
    say(f"csrmm {n} rows of {mean} ncols={ncols} {np.dtype(dtype).name}")
    rng = np.random.default_rng(n)
    lens = rng.integers(0, 2 * mean + 1, n)
    lens[0] = 11 * mean
    _check(lens, 1500, ncols, dtype, -0.75, 0.5)
