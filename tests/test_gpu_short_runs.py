"""Runs that an iteration limit ends cost what their iterations cost, not a
whole chunk of captured ones: the limit's share of a chunk of 64 (8 in
multigrid), with room for what every call pays (the right-hand side, the
read-back)."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

W = {"dxx": 0.1, "dyy": 0.1, "dzz": 0.1, "dxy": 0.1, "dxz": 0.1, "dyz": 0.1,
     "dx": 1.0, "dy": 1.0, "dz": 1.0}


@pytest.mark.parametrize("solver", ["fp64", "fp32", "lsmr", "mg"])
def test_short_runs_against_a_chunk(solver):
    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    nn = (128, 128, 128)
    n = int(np.prod(nn))
    s = fs.FdSystem(_lib.make_grid((0, 0, 0), (1 / 127,) * 3, nn), fs.reg_struct(W, nn, 1e-4))
    p = torch.rand((500, 5), dtype=fs.F64, device="cuda")
    s.set_rows(fs.build_rows(s.grid, _lib.ROWS_VALUE, p, 4, 1.0, n))

    def run(maxiter):
        if solver == "lsmr":
            return s.lsmr(atol=0.0, btol=0.0, conlim=0.0, maxiter=maxiter)[1]["iterations"]
        if solver == "mg":
            return s.solve(rtol=0.0, maxiter=maxiter, multigrid=True)[1]["iterations"]
        return s.solve(rtol=0.0, maxiter=maxiter, precision=solver, inner_rtol=1e-30,
                       max_outer=1)[1]["iterations"]

    best = {}
    few, chunk = (1, 8) if solver == "mg" else (2, 64)
    for maxiter in (few, chunk):
        best[maxiter] = np.inf
        for _ in range(6):
            torch.cuda.synchronize()
            t = time.perf_counter()
            assert run(maxiter) == maxiter
            torch.cuda.synchronize()
            best[maxiter] = min(best[maxiter], time.perf_counter() - t)
    assert best[few] <= 0.3 * best[chunk], best
    s.close()
