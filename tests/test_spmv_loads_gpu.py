"""SpMV with metadata on both sides of the sizes at which the way its entries are read
changes (24 and 192 MB of values and columns, in FP64 24, 64 and 128; with extended precision also rows shorter
and longer than 12): the oracle's bars, and the same bits from two calls. Rows of 20 and
30 with parts of other lengths, so that few blocks are row-wise."""
import numpy as np
import pytest

from gpu_helpers import row_tolerance, rp_from_lengths, say, spmv_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [False, True], ids=["plain", "extended"])
@pytest.mark.parametrize("dtype,nnz", [(np.float64, 2_050_000), (np.float64, 2_150_000), (np.float32, 3_100_000),
                                       (np.float64, 5_500_000), (np.float64, 5_700_000),
                                       (np.float32, 3_200_000), (np.float64, 11_100_000), (np.float64, 11_250_000),
                                       (np.float32, 25_100_000), (np.float32, 25_250_000)])
def test_long_rows(dtype, nnz, ext):
    mb = nnz * (4 + np.dtype(dtype).itemsize) / 2 ** 20
    assert min(abs(mb - k) for k in (24, 64, 128, 192)) < 2
    say(f"spmv with metadata, {mb:.0f} MB of entries, {np.dtype(dtype).name} ext={ext}")
    rng = np.random.default_rng(nnz)
    lengths = np.concatenate([np.full(nnz // 100, 20), np.full(3, 5000), np.full(7, 1500)])
    lengths = np.concatenate([lengths, np.full((nnz - lengths.sum()) // 30, 30)])
    lengths = np.append(lengths, nnz - lengths.sum())
    rp = rp_from_lengths(lengths)
    m = 50000
    ci = rng.integers(0, m, nnz, dtype=np.uint32)
    v = rng.uniform(-1, 1, nnz)
    out = [spmv_check(rp, ci, v, m, dtype, alpha=-0.75, beta=0.5, ext=ext, tol=row_tolerance(rp, dtype))[1]
           for _ in range(2)]
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("dtype,nnz", [(np.float64, 2_050_000), (np.float64, 3_000_000), (np.float32, 3_000_000),
                                       (np.float32, 4_000_000)])
def test_short_rows(dtype, nnz):
    say(f"extended spmv with metadata, short rows, {nnz} entries, {np.dtype(dtype).name}")
    rng = np.random.default_rng(nnz)
    rp = rp_from_lengths(rng.integers(0, 11, nnz // 5))
    m = 50000
    ci, v = rng.integers(0, m, rp[-1]).astype(np.uint32), rng.uniform(-1, 1, rp[-1])
    out = [spmv_check(rp, ci, v, m, dtype, ext=True, tol=row_tolerance(rp, dtype))[1] for _ in range(2)]
    np.testing.assert_array_equal(out[0], out[1])
