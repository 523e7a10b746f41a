"""SpMV without metadata on both sides of its rules: lanes per row (2 to 64 by the mean
row length) with rows at the lengths where the wave (16 times the lanes) and the
workgroup (2048) take them over, many of those in one workgroup; windows of rows
(matrices of 4 M entries and more in rows of fewer than 128) at the lengths of a block
(512) and of a shared row (8192), more of those in one window than its list holds.
Bars of test_spmv_gpu.py; two calls give the same bits."""
import numpy as np
import pytest

from gpu_helpers import random_csr, row_tolerance, rp_from_lengths, say, spmv_check

pytestmark = pytest.mark.gpu


def _check(rp, ci, v, m, dtype, alpha, beta, ext):
    out = [spmv_check(rp, ci, v, m, dtype, alpha=alpha, beta=beta, adaptive=False, ext=ext,
                      tol=row_tolerance(rp, dtype))[1] for _ in range(2)]
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("ext", [False, True], ids=["plain", "extended"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lanes,mean", [(2, 1), (4, 5), (8, 10), (16, 20), (32, 40), (64, 100)])
def test_lanes_per_row(lanes, mean, dtype, ext):
    say(f"spmv rows {lanes} lanes {np.dtype(dtype).name} ext={ext}")
    rng = np.random.default_rng(lanes)
    edge = np.array([16 * lanes - 1, 16 * lanes, 16 * lanes + 1, 2047, 2048, 2049, 5000, 0, 0, 64, 63])
    n = 60 * edge.sum() // mean  # the edges do not move the mean
    lengths = np.maximum(rng.integers(0, 2 * mean + 1, n), 1 if mean == 1 else 0)
    at = rng.choice(n, edge.size, replace=False)
    lengths[at] = edge
    lengths[-1] = 3000              # in the last, part-filled workgroup
    lengths[1000:1012] = 2100       # more than one shared row in a workgroup
    m = 20000
    rp = rp_from_lengths(lengths)
    assert {1: 2, 5: 4, 10: 8, 20: 16, 40: 32, 100: 64}[mean] == lanes and rp[-1] < 4_000_000
    got = int(rp[-1]) // n
    assert {2: got < 4, 4: 4 <= got < 8, 8: 8 <= got < 16, 16: 16 <= got < 32, 32: 32 <= got < 64, 64: got >= 64}[lanes]
    ci = rng.integers(0, m, rp[-1]).astype(np.uint32)
    v = rng.uniform(-1, 1, rp[-1])
    _check(rp, ci, v, m, dtype, -0.75, 0.5, ext)


@pytest.mark.parametrize("ext", [False, True], ids=["plain", "extended"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mean", [6, 24, 100, 120])
def test_windows(mean, dtype, ext):
    say(f"spmv windows of mean {mean} {np.dtype(dtype).name} ext={ext}")
    rng = np.random.default_rng(mean)
    n = 4_600_000 // mean
    lengths = rng.integers(0, 2 * mean + 1, n)
    edge = np.array([511, 512, 513, 0, 0, 1023, 1025, 8191, 8192, 8193, 20000, 1])
    lengths[rng.choice(n - 1, edge.size, replace=False)] = edge
    lengths[64:76] = 8300           # twelve shared rows in one window
    lengths[-1] = 700               # in the last, part-filled window
    m = 30000
    rp = rp_from_lengths(lengths)
    assert rp[-1] >= 4_000_000 and rp[-1] // n < 128
    ci = rng.integers(0, m, rp[-1]).astype(np.uint32)
    v = rng.uniform(-1, 1, rp[-1])
    _check(rp, ci, v, m, dtype, 1.0, 0.0, ext)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_long_rows_of_a_large_matrix(dtype):
    """Rows of 128 entries on average keep the lanes per row, also above 4 M entries."""
    say(f"spmv rows of a large matrix {np.dtype(dtype).name}")
    rng = np.random.default_rng(9)
    rp, ci, v = random_csr(rng, np.concatenate([np.full(20000, 220), [30000, 1, 0, 1025]]), 40000)
    _check(rp, ci, v, 40000, dtype, 1.0, 0.5, False)


@pytest.mark.parametrize("pad", [1, 3])
def test_row_pointer_past_zero_and_no_rows_past_the_end(pad):
    say(f"spmv without metadata, row pointer starts at {pad}")
    rng = np.random.default_rng(6)
    rp = rp_from_lengths(rng.integers(0, 16, 600_000))
    ci, v = rng.integers(0, 900, rp[-1]).astype(np.uint32), rng.uniform(-1, 1, rp[-1])
    assert rp[-1] >= 4_000_000
    rp2 = (rp + pad).astype(np.uint32)
    ci2 = np.concatenate([np.zeros(pad, np.uint32), ci])
    v2 = np.concatenate([np.full(pad, np.nan), v])
    spmv_check(rp2, ci2, v2, 900, np.float64, adaptive=False, tol=row_tolerance(rp2, np.float64))
