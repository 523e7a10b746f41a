"""FP64 reductions of every length add in one order: chains of (up to 16,384
elements) eight elements per lane of ceil(n / 2048) groups of 256 lanes, neighbours
pairwise within 64 lanes, the four waves of a group one after the other, and the
groups' sums pairwise again. Formed here by numpy, the results are the same bits,
on both sides of the length up to which one workgroup does all."""
import ctypes

import numpy as np
import pytest
import torch

import clsparse_amd as cls
from gpu_helpers import say

pytestmark = pytest.mark.gpu


def _pairwise(s):
    while s.shape[-1] > 1:
        s = s[..., 0::2] + s[..., 1::2]
    return s[..., 0]


def _ordered_sum(x):
    g = max(1, -(-x.size // 2048))
    chains = np.zeros(g * 256)
    for i in range(0, x.size, g * 256):
        part = x[i:i + g * 256]
        chains[:part.size] += part
    waves = _pairwise(chains.reshape(g, 4, 64))
    groups = ((waves[:, 0] + waves[:, 1]) + waves[:, 2]) + waves[:, 3]
    assert g <= 64
    return _pairwise(np.concatenate([groups, np.zeros(64 - g)]))


@pytest.mark.parametrize("n", [1, 65, 257, 1024, 2048, 2049, 6000, 8192, 8193, 10000, 14337, 16383, 16384, 16385,
                               60000])
def test_sums_are_the_same_bits(n):
    say(f"order of the reductions, n={n}")
    x = np.random.default_rng(n).uniform(-1, 1, n)
    lib = cls.load()
    with cls.Control() as ctl:
        xd = cls.DenseVector(torch.tensor(x, device="cuda"))
        out = torch.zeros(1, dtype=torch.float64, device="cuda")
        sc = cls.Scalar(out)
        for name, terms in (("reduce", x), ("nrm1", np.abs(x))):
            assert getattr(lib, f"cldenseD{name}")(ctypes.byref(sc.s), ctypes.byref(xd.s), ctl.handle) == 0
            torch.cuda.synchronize()
            assert out.item() == _ordered_sum(terms), name
