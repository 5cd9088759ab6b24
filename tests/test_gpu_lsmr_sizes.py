"""Fixed runs of the LSMR kernels at the edges of their launches, against
scipy's lsmr on the oracle's explicit system.

Sizes: less than one workgroup; no data rows but one; a grid whose partials are
summed in launches of their own (more than 2048 workgroups of 256 nodes);
odd and even step counts, one and more than a chunk of two (the state alternates
between two slots).  Bar: 1e-12 relative after at most 10 steps, where two row
orders of scipy's own lsmr differ by about 1e-15.
"""
import numpy as np
import pytest

from test_gpu_lsmr import _interp, _scipy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,nv,steps,every", [
    (2, 9, 1, 64), (5, 1, 3, 2), (6, 400, 4, 1), (9, 70000, 5, 3), (81, 300, 10, 4),
])
def test_fixed_runs_match_scipy(cells, nv, steps, every):
    rng = np.random.default_rng(cells)
    pts = rng.uniform(0.02, 0.98, (nv, 3))
    values = np.c_[pts, pts @ [0.3, -0.2, 0.9] + 0.1 * rng.normal(size=nv), np.ones(nv)]
    fixed = {"atol": 0.0, "btol": 0.0, "conlim": 0.0, "maxiter": steps}
    it = _interp(cells, values, None, regularisation=0.1)
    assert it.solve_system("lsmr", solver_kwargs=dict(fixed))
    want, istop, itn, _ = _scipy(cells, {"value": values}, **fixed)
    assert (istop, itn) == (7, steps)
    again, info = it._build_system()[0].lsmr(atol=0.0, btol=0.0, conlim=0.0, maxiter=steps,
                                  check_every=every)
    assert (info["istop"], info["iterations"]) == (7, steps)
    for got in (it.c, again.cpu().numpy()):
        assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want)
