"""Weights of uniform families: statistics of the setup report, stored entries."""
import numpy as np
import pytest
import torch

import loopstructural_amd as L
from loopstructural_amd.interpolators import _weight_statistics


@pytest.mark.parametrize("parts", [
    [np.array([1.0, 2.0, 5.0])], [(0.1, 7)], [(0.1, 7), (0.3, 1)],
    [np.array([2.0]), (0.5, 4), np.array([0.1, 9.0])]])
def test_matches_the_arrays(parts):
    w = np.concatenate([p if isinstance(p, np.ndarray) else np.full(p[1], p[0]) for p in parts])
    mean, lo, hi = _weight_statistics(parts)
    assert lo == w.min() and hi == w.max()
    assert mean == pytest.approx(w.mean(), rel=1e-14)


def test_report_follows_the_weights_in_force():
    """The scale may be switched on after the rows were set up."""
    support = L.StructuredGrid(origin=np.zeros(3), nsteps=np.array([5, 6, 7]),
                               step_vector=np.ones(3))
    interp = L.FiniteDifferenceInterpolator(support)
    interp.assemble_borders()
    scale = np.linspace(1.0, 2.0, support.n_nodes)
    for on in (False, True):
        interp.use_regularisation_weight_scale = on
        interp._regularisation_scale = torch.from_numpy(scale)
        w = np.concatenate([c["w"] for c in interp.constraints.values()])
        fam = interp.finalize_setup_diagnostics_report().families["regularisation"]
        assert (fam.effective_weight_min, fam.effective_weight_max) == (w.min(), w.max())
        assert fam.effective_weight_mean == pytest.approx(w.mean(), rel=1e-14)
    assert w.max() > w.min()


@pytest.mark.parametrize("read", [
    lambda c: dict(c.items())["w"], lambda c: list(c.values())[list(c).index("w")],
    lambda c: dict.__getitem__(c.copy(), "w"), lambda c: c.pop("w"), lambda c: c.raw("w"),
    lambda c: c["w"]])
def test_edge_jump_weights_are_an_array(read):
    """However the entry is read, and once it has been, the same array."""
    mesh = L.TetMesh(origin=np.zeros(3), nsteps=np.array([3, 3, 3]), step_vector=np.ones(3))
    interp = L.P1Interpolator(mesh)
    interp.minimise_edge_jumps(0.3)
    con = interp.constraints["edge jump"]
    w = read(con)
    assert isinstance(w, np.ndarray) and w.shape == con["b"].shape and (w == 0.3).all()
    assert "w" not in con or con["w"] is w
