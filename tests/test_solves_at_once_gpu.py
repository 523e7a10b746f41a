"""Solves of several threads at once, each with its own control and stream, on the
sizes that share the chip (few workgroups) and those that take all of it: the same
bits as one after the other."""
import threading

import numpy as np
import pytest
import torch

import clsparse_amd as cls
from gpu_helpers import cg_call, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(30, 31), (93, 101), (64, 64, 60), (100, 90, 110)])
def test_threads_give_the_bits_of_single_solves(shape):
    say(f"concurrent solves {shape}")
    rp, ci, v, m = (cls.gen_poisson2d(*shape) if len(shape) == 2 else
                    cls.gen_diffusion3d(*shape, sigma=1.0, ax=1.0, ay=1.0, az=1.0, seed=2))[:4]
    torch.cuda.init()

    def solve(seed, out, start=None):
        with torch.cuda.stream(torch.cuda.Stream()), cls.Control() as ctl:
            A = cls.CsrMatrix(rp, ci, v, m)
            A.meta_create(ctl)
            b = torch.tensor(cls.gen_uniform(m, -1, 1, seed=seed), device="cuda")
            if start is not None:
                start.wait(30)
            for _ in range(3):
                x = torch.zeros_like(b)
                sc = cls.SolverControl(cls.DIAGONAL, 2000, 1e-8, 0.0)
                status = cg_call(A, x, b, sc, ctl)
                st, n = sc.stats(), sc.launches()
                sc.release()
                out.append((status, st.status_detail, n.gave_up + n.refused, st.n_iters, x.cpu().numpy()))

    alone = {}
    for seed in (1, 2, 3, 4):
        solve(seed, alone.setdefault(seed, []))
    together, barrier = {seed: [] for seed in alone}, threading.Barrier(len(alone))
    threads = [threading.Thread(target=solve, args=(seed, together[seed], barrier)) for seed in alone]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    for seed, runs in alone.items():
        assert len(together[seed]) == len(runs) == 3
        for one, many in zip(runs, together[seed]):
            assert one[:4] == many[:4] and one[:3] == (0, 0, 0)
            np.testing.assert_array_equal(one[4], many[4])
