"""Memory of the Jacobi PCG's data term by node: who holds it, how much of it,
and what happens without it.

The bounds: rows of W entries (16 or 32) of 4 bytes of column and 8 or 4 of
value per data node, a quarter more for the next row set, and SLACK for what
the runtime itself takes (captured graphs, whole pages)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

W = {"dxx": 0.1, "dyy": 0.1, "dzz": 0.1, "dxy": 0.1, "dxz": 0.1, "dyz": 0.1,
     "dx": 1.0, "dy": 1.0, "dz": 1.0}
NODES = (58, 56, 54)
SLACK = 6 << 20


def _grid():
    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    return (_lib.make_grid((0, 0, 0), tuple(1.0 / (k - 1) for k in NODES), NODES),
            fs.reg_struct(W, NODES, 1e-4), int(np.prod(NODES)))


def _single_node_rows(n, count):
    """One entry per row, every row at a node of its own."""
    from loopstructural_amd import fd_system as fs

    dev = torch.device("cuda")
    at = torch.linspace(0, n - 1, count, device=dev).long()
    one = torch.ones(count, dtype=fs.F64, device=dev)
    return fs.FdRows(torch.arange(count + 1, device=dev), at.to(torch.int32), one,
                     torch.cos(at.to(fs.F64)), one.clone(), one.clone(), n)


def _taken(fn):
    """Device memory that a call leaves behind."""
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    out = fn()
    torch.cuda.synchronize()
    return free - torch.cuda.mem_get_info()[0], out


def test_batch_solves_take_none():
    from loopstructural_amd import fd_system as fs

    g, reg, n = _grid()
    bs = fs.BatchSystem([g, g], reg)
    for count in (10, 100_000):
        rows = _single_node_rows(n, count)
        bs.set_rows([rows, rows])
        taken, _ = _taken(lambda: bs.solve(rtol=1e-3, maxiter=8, precision="fp32"))
    assert taken <= SLACK, taken
    bs.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_solve_without_room_for_them(monkeypatch, precision):
    """The allocation fails on one handle and not on another: both solve, to
    the same field, and nothing stays behind; the next row set tries again."""
    from loopstructural_amd import fd_system as fs

    g, reg, n = _grid()
    kw = {"rtol": 1e-9, "precision": precision}
    fields = []
    for fail in (True, False):
        s = fs.FdSystem(g, reg)
        s.set_rows(_single_node_rows(n, 10))
        s.solve(**kw)
        s.set_rows(_single_node_rows(n, 60_000))
        if fail:
            monkeypatch.setenv("LSAMD_FAULT_INJECT", "node_rows")
        taken, (c, info) = _taken(lambda: s.solve(**kw))
        monkeypatch.delenv("LSAMD_FAULT_INJECT", raising=False)
        assert info["converged"]
        fields.append(c)
        assert (taken <= SLACK) == fail, (fail, taken)
        if fail:
            s.set_rows(_single_node_rows(n, 59_000))
            taken, (_, info) = _taken(lambda: s.solve(**kw))
            assert info["converged"] and taken > SLACK
        s.close()
    err = float((fields[0] - fields[1]).norm() / fields[1].norm())
    assert err <= 1e-6, err


def test_memory_is_that_of_the_width_and_the_precision():
    """Rows of 16 entries; FP64, then FP32 beside it, then the other way round
    on a second handle; the fields agree with a multigrid solve (which builds
    both in one pass)."""
    from loopstructural_amd import fd_system as fs

    g, reg, n = _grid()
    count = 60_000
    col, v64, v32 = (1.25 * 16 * k * count for k in (4, 8, 4))
    per_node = 1.25 * 8 * count + n  # the product's compact result, partials, masks
    fields = []
    for order in (("fp64", "fp32"), ("fp32", "fp64"), ("mg",)):
        s = fs.FdSystem(g, reg)
        run = {p: (lambda p=p: s.solve(rtol=1e-9, precision=p)) for p in ("fp64", "fp32")}
        run["mg"] = lambda: s.solve(rtol=1e-9, multigrid=True)
        s.set_rows(_single_node_rows(n, 10))
        for p in order:
            run[p]()
        s.set_rows(_single_node_rows(n, count))
        for first, p in zip((True, False), order):
            taken, (c, info) = _taken(run[p])
            assert info["converged"]
            fields.append(c)
            if p != "mg":
                room = (v32 if p == "fp32" else v64) + (col + per_node if first else 0)
                assert taken <= room + SLACK, (order, p, taken, room)
        s.close()
    for c in fields[:-1]:
        assert float((c - fields[-1]).norm() / fields[-1].norm()) <= 1e-6


@pytest.mark.parametrize("multigrid,count", [(False, 60_000), (False, 60_001), (True, 137_500),
                                             (True, 137_501)])
def test_many_data_nodes_take_the_row_form(monkeypatch, multigrid, count):
    """At and past the limits (50000 + entries / 6 data nodes in the Jacobi
    solve, 110000 + entries / 5 in multigrid): node rows on one side only, and
    the iterates of the row form either way.  Nine steps; their rounding differs
    by the order of the sums: FP64 (2^-53, a few hundred of them) in the Jacobi
    solve; in multigrid also in the FP32 V-cycle, whose every output may differ by
    some 2^-24 = 6e-8 of itself, and an iterate by no more than that share of
    its size for each of the nine directions."""
    from loopstructural_amd import fd_system as fs

    g, reg, n = _grid()
    s = fs.FdSystem(g, reg)
    kw = {"rtol": 0.0, "maxiter": 9, "multigrid": multigrid}
    s.set_rows(_single_node_rows(n, 10))
    s.solve(**kw)
    rows = _single_node_rows(n, count)
    if multigrid:  # the hierarchy's memory apart
        s.set_rows(rows)
        monkeypatch.setenv("LSAMD_FAULT_INJECT", "node_rows")
        s.solve(**kw)
        monkeypatch.delenv("LSAMD_FAULT_INJECT")
    s.set_rows(rows)
    taken, (c, _) = _taken(lambda: s.solve(**kw))
    assert (taken > SLACK) == (count % 10 == 0), taken
    monkeypatch.setenv("LSAMD_FAULT_INJECT", "node_rows")
    s.set_rows(rows)
    want, _ = s.solve(**kw)
    assert float((c - want).norm() / want.norm()) <= (9 * 6e-8 if multigrid else 1e-11)
    s.close()


def test_rows_of_a_weighted_p1_regulariser_take_none():
    """Nine rows per node, as a P1 regulariser with weights of its own gives:
    no memory for node rows; a quarter of the rows has them.  The iterates of
    the row form either way (FP64, a few hundred terms per sum)."""
    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    nn = (30, 28, 26)
    n, dev = int(np.prod(nn)), torch.device("cuda")
    g = _lib.make_grid((0, 0, 0), tuple(1.0 / (k - 1) for k in nn), nn)
    gen = torch.Generator(device=dev).manual_seed(1)
    corner = torch.tensor([i + nn[0] * (j + nn[1] * k) for k in (0, 1) for j in (0, 1)
                           for i in (0, 1)], device=dev)
    for m, some in ((9 * n, False), (9 * n // 4, True)):
        at = torch.arange(m, device=dev) % n
        one = torch.ones(m, dtype=fs.F64, device=dev)
        rows = fs.FdRows(torch.arange(m + 1, device=dev) * 8,
                         (at[:, None] + corner).clamp(max=n - 1).reshape(-1).to(torch.int32),
                         torch.rand(8 * m, dtype=fs.F64, device=dev, generator=gen) - 0.4,
                         torch.cos(one.cumsum(0)), one, one.clone(), n)
        s = fs.P1System(g, 0.1, 1e-2)
        s.set_rows(_single_node_rows(n, 10))
        s.solve(rtol=0.0, maxiter=6)
        s.set_rows(rows)
        taken, (c, _) = _taken(lambda: s.solve(rtol=0.0, maxiter=6))
        assert (taken > 5 << 20) == some, taken  # 22e3 x 32 entries x 12 bytes: 8 MiB
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("LSAMD_FAULT_INJECT", "node_rows")
            s.set_rows(rows)
            want, _ = s.solve(rtol=0.0, maxiter=6)
        assert float((c - want).norm() / want.norm()) <= 1e-11
        s.close()
