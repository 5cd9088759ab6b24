"""Evaluation and P1 location where their short cuts could differ from the
oracle: steps and origins of every scale (known divisors, the plain divisions
beyond them, the tet preselection and its fall-back), points on nodes, edges
and faces, tiny coordinates, and partial workgroups."""
import numpy as np
import pytest
import torch

from oracle import fd as ofd
from oracle import p1 as op1

pytestmark = pytest.mark.gpu

GRIDS = [
    ((0.0, 0.0, 0.0), (7, 5, 6), (1 / 7, 0.2, 1 / 6)),
    ((512345.25, 7654321.5, -3000.0), (12, 9, 8), (37.5, 41.3, 11.7)),  # projected metres
    ((-1e6, 3.0, 0.0), (6, 5, 4), (1e-3, 250.0, 3.0)),   # positions far coarser than the step
    ((1e9, 0.0, 0.0), (5, 4, 6), (1e-5, 1.0, 1.0)),      # past the preselection's slack
    ((0.0, 0.0, 0.0), (5, 6, 4), (1e-70, 1.0, 2.0)),     # a step that is no known divisor
    ((0.0, 0.0, 0.0), (3, 4, 5), (0.25, 0.5, 0.125)),
]


def _points(o, cells, h, n, seed):
    rng = np.random.default_rng(seed)
    o, h, cells = np.array(o), np.array(h), np.array(cells)
    ext = h * cells
    p = o + rng.uniform(-0.05, 1.05, (n, 3)) * ext
    q = o + h * rng.integers(0, cells + 1, (n, 3))           # nodes
    e = p.copy()                                             # edges and faces
    on = rng.random((n, 3)) < 0.5
    e[on] = q[on]
    d = q + h * rng.choice([0.0, 0.25, 0.5, 0.75], (n, 3))   # diagonals, tet faces
    tiny = p.copy()
    tiny[:, rng.integers(0, 3)] = o[0] + 1e-300
    near = q * (1 + rng.choice([-2e-16, 0, 2e-16], (n, 3)))
    return np.vstack([p, q, e, d, tiny, near])


def _grid(o, cells, h):
    from loopstructural_amd import _lib

    return _lib.make_grid(o, h, np.array(cells) + 1)


@pytest.mark.parametrize("gi", range(len(GRIDS)))
def test_fd_bit_exact(gi):
    from loopstructural_amd import fd_system as fs

    o, cells, h = GRIDS[gi]
    og = ofd.Grid(o, cells, h)
    pts = _points(o, cells, h, 700, gi)
    c = np.random.default_rng(gi).standard_normal(og.n_nodes)
    with np.errstate(all="ignore"):
        rv, rg = ofd.evaluate_value(og, c, pts), ofd.evaluate_gradient(og, c, pts)
    for n in (1, 255, 256, 257, len(pts)):
        v, g = fs.evaluate(_grid(o, cells, h), torch.from_numpy(c), torch.from_numpy(pts[:n]),
                           True, True)
        assert np.array_equal(v.cpu().numpy(), rv[:n], equal_nan=True)
        assert np.array_equal(g.cpu().numpy(), rg[:n], equal_nan=True)
    v, _ = fs.evaluate(_grid(o, cells, h), torch.from_numpy(c), torch.from_numpy(pts), True, False)
    assert np.array_equal(v.cpu().numpy(), rv, equal_nan=True)


@pytest.mark.parametrize("gi", range(len(GRIDS)))
def test_p1_bit_exact(gi):
    from loopstructural_amd import fd_system as fs

    o, cells, h = GRIDS[gi]
    m = op1.TetMesh(o, cells, h)
    pts = _points(o, cells, h, 700, 50 + gi)
    c = np.random.default_rng(gi).standard_normal(m.n_nodes)
    with np.errstate(all="ignore"):
        _, bc, tet, ins = m.element_for_location(pts)
        rv, rg = m.evaluate_value(pts, c), m.evaluate_gradient(pts, c)
    gt, _, gi_, gb, _ = fs.p1_locate(_grid(o, cells, h), torch.from_numpy(pts))
    assert np.array_equal(gi_.cpu().numpy(), ins)
    assert np.array_equal(gt.cpu().numpy()[ins], tet[ins])
    assert np.array_equal(gb.cpu().numpy()[ins], bc[ins])
    for n in (1, 255, 256, 257, len(pts)):
        v, g = fs.p1_evaluate(_grid(o, cells, h), torch.from_numpy(c), torch.from_numpy(pts[:n]),
                              True, True)
        assert np.array_equal(v.cpu().numpy(), rv[:n], equal_nan=True)
        g, r = g.cpu().numpy(), rg[:n]
        assert np.array_equal(np.isnan(g), np.isnan(r))
        # the oracle's gradient is a sum of four corner terms |c| / h: a few
        # roundings of the largest
        scale = np.abs(c).max() / (np.array(h))
        assert np.all(np.nan_to_num(np.abs(g - r) / scale) <= 1e-14)
