"""Rounding of the FP64 SpMV without metadata on a matrix of 4.3 M entries, whose
rows' entries are multiplied into LDS and added there.

With values and x in [0, 1] a row of 16 products sums to about 4. Its products'
roundings (each at most 2^-53 of its product, independent) and one rounding of
the sum have a root mean square of at most 2^-53 / sqrt(3) (1 + 1 / 16)^(1/2) of
the sum: 0.6 2^-53. Adding the 16 rounded products one after the other has 2^-53 /
sqrt(3) (sum over k of (k / 16)^2)^(1/2) besides, 1.4 2^-53 at most and in the
mean over a binade 0.9 2^-53."""
import numpy as np
import pytest
import torch

import clsparse_amd as cls
from gpu_helpers import U64, say

pytestmark = pytest.mark.gpu

N, K = 270_000, 16


def _matrix(rng):
    rp = (np.arange(N + 1) * K).astype(np.uint32)
    ci = np.sort(rng.integers(0, N, (N, K)), axis=1).astype(np.uint32)
    return rp, ci, rng.uniform(0, 1, (N, K)), rng.uniform(0, 1, N)


def _run(rp, ci, v, x):
    with cls.Control() as ctl:
        A = cls.CsrMatrix(rp, ci.ravel(), v.ravel(), N)
        y = cls.DenseVector(torch.full((N,), float("nan"), dtype=torch.float64, device="cuda"))
        cls.check("csrmv", A.spmv(cls.Scalar(1.0), cls.DenseVector(torch.tensor(x, device="cuda")), cls.Scalar(0.0), y,
                                  ctl))
        return y.t.cpu().numpy()


def test_rows_are_rounded_once_beside_their_products():
    say("spmv without metadata: rounding of 16-entry rows")
    rp, ci, v, x = _matrix(np.random.default_rng(11))
    y = _run(rp, ci, v, x)
    exact = (v.astype(np.longdouble) * x[ci]).sum(axis=1)
    rel = ((y - exact) / exact).astype(np.float64)
    assert np.sqrt((rel ** 2).mean()) <= 0.6 * U64


def test_infinite_sums_stay_infinite():
    """A compensated sum's error term is NaN where the sum is infinite."""
    say("spmv without metadata: infinities and NaN")
    rp, ci, v, x = _matrix(np.random.default_rng(12))
    v[5, 3], v[6, 0], v[7, 15] = np.inf, -np.inf, np.nan
    v[8, 2], v[8, 9] = np.inf, -np.inf
    v[9] = 1e308 / x[ci[9]]  # finite products whose sum overflows
    y = _run(rp, ci, v, x)
    assert y[5] == np.inf and y[6] == -np.inf and np.isnan(y[7]) and np.isnan(y[8]) and y[9] == np.inf
    assert np.isfinite(np.delete(y, [5, 6, 7, 8, 9])).all()
