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


@pytest.mark.parametrize("nn,n,kind", [
    ((128, 128, 64), 1 << 22, "random"),     # the smallest grid and list with a table
    ((131, 97, 83), (1 << 22) + 37, "random"),
    ((131, 97, 83), (1 << 22) + 37, "ordered"),
    ((131, 97, 83), (1 << 22) + 37, "mixed"),
    ((128, 128, 63), 1 << 22, "random"),     # one plane less: none
])
def test_fd_corner_table_changes_nothing(nn, n, kind):
    """Evaluation with scratch memory against the one without, bit for bit,
    and a piece of it against the oracle."""
    import ctypes as C

    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    o, h = (10.0, -3.0, 0.5), (0.25, 0.5, 0.125)
    cells = np.array(nn) - 1
    rng = np.random.default_rng(n % 1000)
    pts = np.array(o) + rng.uniform(-0.01, 1.01, (n, 3)) * cells * h
    if kind != "random":
        pts = pts[np.argsort(pts[:, 2], kind="stable")]
        pts[:, 0] = o[0] + np.linspace(0.1, 0.9, n) * cells[0] * h[0]
        pts[:, 1] = o[1] + 0.3 * cells[1] * h[1]
    if kind == "mixed":
        pts[n // 2:] = np.array(o) + rng.random((n - n // 2, 3)) * cells * h
    pts[::100003] = np.nan
    pts[7::100003] = np.array(o) + cells * h
    c = rng.standard_normal(int(np.prod(nn)))
    grid = _grid(o, cells, h)
    size = C.c_int64(0)
    _lib.call("lsamd_fd_evaluate_scratch", C.byref(grid), n, C.byref(size))
    assert size.value == (0 if nn[2] == 63 else 8 * (16 + 4 * c.size))
    dc, dp = torch.from_numpy(c).cuda(), torch.from_numpy(pts).cuda()
    v, g = fs.evaluate(grid, dc, dp, True, True)
    v0, g0 = torch.empty_like(v), torch.empty_like(g)
    _lib.call("lsamd_fd_evaluate", C.byref(grid), _lib.ptr(dc), _lib.ptr(dp), n, _lib.ptr(v0),
              _lib.ptr(g0), _lib.stream())
    assert torch.equal(v.view(torch.int64), v0.view(torch.int64))
    assert torch.equal(g.view(torch.int64), g0.view(torch.int64))
    part = slice(0, 5000)
    og = ofd.Grid(o, tuple(int(x) for x in cells), h)
    with np.errstate(all="ignore"):
        assert np.array_equal(v[part].cpu().numpy(), ofd.evaluate_value(og, c, pts[part]),
                              equal_nan=True)
        assert np.array_equal(g[part].cpu().numpy(), ofd.evaluate_gradient(og, c, pts[part]),
                              equal_nan=True)
    only, _ = fs.evaluate(grid, dc, dp, True, False)
    assert torch.equal(only.view(torch.int64), v0.view(torch.int64))
    _, only = fs.evaluate(grid, dc, dp, False, True)
    assert torch.equal(only.view(torch.int64), g0.view(torch.int64))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("support", ["fd", "p1"])
def test_coefficients_that_are_not_finite(support, bad):
    """A NaN or infinite coefficient reaches every value and every gradient
    component that the sum over the cell's or the tet's corners gives it, and
    no other point."""
    from loopstructural_amd import fd_system as fs

    o, cells, h = GRIDS[0]
    og = ofd.Grid(o, cells, h) if support == "fd" else op1.TetMesh(o, cells, h)
    pts = np.array(o) + np.random.default_rng(5).uniform(0, 1, (3000, 3)) * np.array(cells) * h
    c = np.random.default_rng(6).standard_normal(og.n_nodes)
    c[::17] = bad
    with np.errstate(all="ignore"):
        if support == "fd":
            rv, rg = ofd.evaluate_value(og, c, pts), ofd.evaluate_gradient(og, c, pts)
        else:
            rv, rg = og.evaluate_value(pts, c), og.evaluate_gradient(pts, c)
    f = fs.evaluate if support == "fd" else fs.p1_evaluate
    v, g = f(_grid(o, cells, h), torch.from_numpy(c), torch.from_numpy(pts), True, True)
    for got, want in ((v.cpu().numpy(), rv), (g.cpu().numpy(), rg)):
        assert 0 < np.isfinite(want).sum() < want.size
        for kind in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(kind(got), kind(want)), kind


@pytest.mark.parametrize("support", ["fd", "p1"])
@pytest.mark.parametrize("gi", [0, 4])
def test_streamed_and_cached_results_are_the_same(gi, support):
    """One call past the last-level cache (256 MiB of points and results), whose
    points are read past it, against calls that fit; steps that are known
    divisors and one that is none."""
    from loopstructural_amd import fd_system as fs

    o, cells, h = GRIDS[gi]
    n = (256 << 20) // 56 + 1
    gen = torch.Generator(device="cuda").manual_seed(gi)
    box = torch.tensor(np.array(cells) * h, device="cuda")
    pts = torch.tensor(o, device="cuda") + torch.rand((n, 3), dtype=fs.F64, device="cuda",
                                                      generator=gen) * box * 1.01
    c = torch.rand(int(np.prod(np.array(cells) + 1)), dtype=fs.F64, device="cuda", generator=gen)
    grid = _grid(o, cells, h)
    f = fs.evaluate if support == "fd" else fs.p1_evaluate
    v, g = f(grid, c, pts, True, True)
    assert 0 < int(torch.isnan(v).sum()) < n
    for part in (slice(0, n // 2), slice(n // 2, n - 1), slice(n - 1, n)):
        v1, g1 = f(grid, c, pts[part], True, True)
        assert torch.equal(v[part].view(torch.int64), v1.view(torch.int64))
        assert torch.equal(g[part].view(torch.int64), g1.view(torch.int64))
