"""Coarse-grid weights of the multigrid preconditioner: the outer iteration
count stays bounded over odd, even and ragged axes, dense and sparse data."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

W = {"dxx": 0.1, "dyy": 0.1, "dzz": 0.1, "dxy": 0.1, "dxz": 0.1, "dyz": 0.1,
     "dx": 1.0, "dy": 1.0, "dz": 1.0}


def make(nodes, n_values, n_normals, seed):
    from loopstructural_amd import _lib, synthetic
    from loopstructural_amd import fd_system as fs

    grid = _lib.make_grid((0, 0, 0), tuple(1.0 / (n - 1) for n in nodes), nodes)
    values, normals = synthetic.constraints(n_values, n_normals, seed)
    s = fs.FdSystem(grid, fs.reg_struct(W, nodes, 1e-8))
    blocks = []
    for pts, kind, wcol, w in ((normals, _lib.ROWS_NORMAL, 6, 10.0 / 3),
                               (values, _lib.ROWS_VALUE, 4, 1.0)):
        p = torch.from_numpy(pts).to(_lib.device())
        _, ins, _, _ = fs.locate(grid, p[:, :3].contiguous(), want_w=False)
        blocks.append(fs.build_rows(grid, kind, p[ins].contiguous(), wcol, w, s.n))
    s.set_rows(fs.concat_rows(blocks, s.n))
    return s


# with weights halved per level these take 80, 85, 100 and 90 iterations
@pytest.mark.parametrize("nodes,n_values,n_normals,most", [
    ((24, 24, 36), 234, 60, 76), ((65, 65, 65), 1000, 200, 80), ((64, 48, 33), 300, 60, 80),
    ((7, 30, 41), 100, 20, 80)])
def test_iterations_and_minimiser(nodes, n_values, n_normals, most):
    s = make(nodes, n_values, n_normals, 77)
    x, info = s.solve(rtol=1e-11, multigrid=True)
    assert info["converged"]
    y, _ = s.solve(rtol=1e-13, precision="fp64")
    assert float(torch.linalg.vector_norm(x - y) / torch.linalg.vector_norm(y)) < 1e-7
    _, info = s.solve(rtol=1e-10, multigrid=True)
    assert info["iterations"] <= most
    s.close()


# extents of a row's columns in fine nodes: on the coarse grid boxes of at most
# 4 nodes (slots) or more (the general form, which takes up to 64 coarse columns)
@pytest.mark.parametrize("extent,entries", [(1, 8), (2, 5), (4, 12), (5, 12), (6, 10), (7, 6),
                                            (30, 3), (5, 1)])
def test_rows_of_any_extent_reach_the_minimiser(extent, entries):
    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    nodes = np.array((34, 33, 41))
    rng = np.random.default_rng(100 * extent + entries)
    nrows, dev = 301, _lib.device()
    lo = rng.integers(0, nodes - extent, (nrows, 1, 3))
    c = lo + rng.integers(0, extent + 1, (nrows, entries, 3))
    cols = c[..., 0] + nodes[0] * (c[..., 1] + nodes[1] * c[..., 2])
    s = fs.FdSystem(_lib.make_grid((0, 0, 0), tuple(1 / (nodes - 1)), nodes),
                    fs.reg_struct(W, tuple(int(n) for n in nodes), 1e-8))
    coef = rng.uniform(0.2, 1.0, (nrows, entries)) / entries
    s.set_rows(fs.FdRows(
        torch.arange(nrows + 1, device=dev) * entries,
        torch.from_numpy(cols.reshape(-1).astype(np.int32)).to(dev),
        torch.from_numpy(coef.reshape(-1)).to(dev), torch.from_numpy(rng.normal(size=nrows)).to(dev),
        torch.ones(nrows, dtype=torch.float64, device=dev), None, s.n))
    x, info = s.solve(rtol=1e-11, multigrid=True)
    assert info["converged"] and info["iterations"] <= 120
    y, _ = s.solve(rtol=1e-13, precision="fp64")
    assert float(torch.linalg.vector_norm(x - y) / torch.linalg.vector_norm(y)) < 1e-7
    s.close()


def test_a_coarse_level_past_a_million_nodes():
    """209^3 nodes: the first coarse level (105^3) keeps the product and smooths
    its covered nodes apart, as the fine level does.  The residual in FP64, by
    the operator and the right-hand side, which other tests compare with the
    oracle; a level that is smoothed wrongly costs iterations."""
    s = make((209, 209, 209), 20000, 3000, 3)
    x, info = s.solve(rtol=1e-10, multigrid=True)
    assert info["converged"] and info["iterations"] <= 90
    scale = torch.sqrt(s.diag())
    r = torch.linalg.vector_norm((s.rhs() - s.apply(x)) / scale)
    assert float(r / torch.linalg.vector_norm(s.rhs() / scale)) <= 1.1e-10
    s.close()


# ridges from one that vanishes beside the other weights to one that rules;
# with weights halved per level these took 78, 103, 113, 28 and 25 iterations
@pytest.mark.parametrize("ridge,most", [(1e-8, 80), (0.01, 85), (0.05, 105), (0.2, 40), (1.0, 33)])
def test_ridge_that_matters(ridge, most):
    from loopstructural_amd import fd_system as fs

    one = make((64, 64, 64), 1500, 300, 1)
    s = fs.FdSystem(one.grid, fs.reg_struct(W, (64, 64, 64), ridge))
    s.set_rows(one.rows)
    x, info = s.solve(rtol=1e-10, multigrid=True)
    assert info["converged"] and info["iterations"] <= most
    y, _ = s.solve(rtol=1e-12, precision="fp64")
    assert float(torch.linalg.vector_norm(x - y) / torch.linalg.vector_norm(y)) < 1e-7
    s.close()
    one.close()
