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
