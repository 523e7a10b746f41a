"""csrmm on matrices of about 2^32 entries, whose last rows end less than a slot's or a
workgroup's step below 2^32 (2^32 - 1 entries: the kernel whose places do not wrap) or
just one step below it (2^32 - 1024: the others). All other rows are empty; the entries
before the last rows' belong to no row. Products of small integers: every sum is exact."""
import ctypes

import numpy as np
import pytest
import torch

import clsparse_amd as cls
from gpu_helpers import say
from test_csrmm_gpu import _dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [2**32 - 1, 2**32 - 1024])
@pytest.mark.parametrize("ncols,lens", [(1, [300, 3, 257]), (8, [5, 256, 300]), (70, [1, 400, 63]), (5, [600, 1100])])
def test_rows_that_end_at_the_last_entry(ncols, lens, nnz):
    if torch.cuda.mem_get_info()[0] + torch.cuda.memory_reserved() < 36 << 30:
        pytest.skip("needs 36 GB of device memory")
    say(f"csrmm {nnz} entries ncols={ncols} rows of {lens}")
    n = 64
    m = 1000
    total = sum(lens)
    rng = np.random.default_rng(ncols)
    col = rng.integers(0, m, total)
    val = rng.integers(-4, 5, total)
    B = rng.integers(-4, 5, (m, ncols))
    ci = torch.zeros(nnz, dtype=torch.int32, device="cuda")
    v = torch.zeros(nnz, dtype=torch.float32, device="cuda")
    ci[nnz - total:] = torch.tensor(col, dtype=torch.int32, device="cuda")
    v[nnz - total:] = torch.tensor(val, dtype=torch.float32, device="cuda")
    rp = torch.empty(n + 1, dtype=torch.int32, device="cuda")
    ends = nnz - total + np.concatenate([[0], np.cumsum(lens)])
    rp.fill_(int(ends[0]) - 2**32)
    rp[n - len(lens):] = torch.tensor(ends - 2**32, dtype=torch.int32, device="cuda")
    Bt = torch.tensor(B.ravel(), dtype=torch.float32, device="cuda")
    Ct = torch.full((n * ncols,), 7.0, dtype=torch.float32, device="cuda")
    A = cls.clsparseCsrMatrix()
    A.num_rows, A.num_cols, A.num_nonzeros = n, m, nnz
    A.values, A.col_indices, A.row_pointer = v.data_ptr(), ci.data_ptr(), rp.data_ptr()
    with cls.Control() as ctl:
        a, b = cls.Scalar(1.0, torch.float32), cls.Scalar(0.0, torch.float32)
        Bd, Cd = _dense(Bt, m, ncols, ncols), _dense(Ct, n, ncols, ncols)
        cls.check("csrmm", cls.load().clsparseScsrmm(ctypes.byref(a.s), ctypes.byref(A), ctypes.byref(Bd),
                                                     ctypes.byref(b.s), ctypes.byref(Cd), ctl.handle))
    C = Ct.reshape(n, ncols)
    assert not C[:n - len(lens)].any()
    want = np.stack([val[s:e] @ B[col[s:e]] for s, e in zip(ends[:-1] - ends[0], ends[1:] - ends[0])])
    np.testing.assert_array_equal(C[n - len(lens):].cpu().numpy(), want)
