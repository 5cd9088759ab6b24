"""Jacobi PCG in its launch forms: the one-launch tile and the direction plus
streaming stencil, the data term by node (both row widths) and by rows.

Fixed numbers of iterations against the oracle's Jacobi PCG on the explicit
normal equations: the iterates of few steps agree to rounding (1e-11), an odd
count stops where it should, and the solve to a tolerance meets it.  The FP32 inner steps are as far from the FP64
iterates as the same recurrence in numpy's float32 is, within a factor of 30
for the orders of the sums (and of the applied matrix, there summed by row)."""
import numpy as np
import pytest
import torch
from scipy import sparse

from oracle import fd as ofd

pytestmark = pytest.mark.gpu

W = {"dxx": 0.1, "dyy": 0.1, "dzz": 0.1, "dxy": 0.1, "dxz": 0.1, "dyz": 0.1,
     "dx": 1.0, "dy": 1.0, "dz": 1.0}


def _rows(n, kind, seed):
    """Random rows: kind 'narrow' (1..4 entries, repeats among them), 'cell'
    (8), 'wide' (one node coupled with 80 others) or 'none'."""
    rng = np.random.default_rng(seed)
    lens = {"narrow": rng.integers(1, 5, 60), "cell": np.full(60, 8),
            "wide": np.r_[np.full(20, 8), 80], "none": np.zeros(0, int)}[kind]
    ptr = np.r_[0, np.cumsum(lens)]
    # columns in a narrow band, so that rows overlap
    cols = (rng.integers(0, n) + rng.integers(0, 60, ptr[-1])) % n
    if kind == "wide":
        cols[ptr[20]:] = rng.permutation(n)[:80]
    # rows of unit length, as every row builder gives them; the error of few
    # iterates then stays near rounding (unnormalised, the one of 80 entries
    # alone stretches the spectrum to 1e7 and seven steps amplify it 1e6 times)
    coef = rng.standard_normal(ptr[-1])
    if len(lens):
        coef /= np.repeat(np.sqrt(np.add.reduceat(coef ** 2, ptr[:-1])), lens)
    return ptr, cols, coef, rng.standard_normal(len(lens)), rng.uniform(0.5, 1.5, len(lens))


def _system(nodes, kind, seed=3):
    from loopstructural_amd import _lib
    from loopstructural_amd import fd_system as fs

    n = int(np.prod(nodes))
    ptr, cols, coef, b, w = _rows(n, kind, seed)
    h = tuple(1.0 / (k - 1) for k in nodes)
    s = fs.FdSystem(_lib.make_grid((0, 0, 0), h, nodes), fs.reg_struct(W, nodes, 1e-4))
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a)).to(s.dev, d)  # noqa: E731
    if len(b):
        s.set_rows(fs.FdRows(t(ptr, torch.int64), t(cols, torch.int32), t(coef, fs.F64),
                             t(b, fs.F64), t(w, fs.F64), t(np.ones(len(b)), fs.F64), n))
    else:
        s.set_rows(None)
    og = ofd.Grid((0, 0, 0), tuple(k - 1 for k in nodes), h)
    N, rhs = ofd.normal_equations(ofd.assemble_fd(og, {}, regularisation=0.1), ridge=1e-4)
    if len(b):
        A = sparse.csr_matrix((coef, cols, ptr), shape=(len(b), n))
        A = sparse.diags(w) @ A
        N, rhs = N + A.T @ A, A.T @ (w * b)
    return s, N.tocsr(), rhs, n


def _pcg32(N, rhs, steps):
    N, r = N.astype(np.float32), rhs.astype(np.float32)
    minv = (1 / N.diagonal()).astype(np.float32)
    x, p = np.zeros_like(r), None
    rho = np.dot(r.astype(float), minv * r)
    for _ in range(steps):
        z = minv * r
        p = z if p is None else z + np.float32(rho / prev) * p
        q = N @ p
        a = np.float32(rho / np.dot(p.astype(float), q))
        x, r, prev = x + a * p, r - a * q, rho
        rho = np.dot(r.astype(float), minv * r)
    return x


# 16 x 8 x 4 tiles: below, at and past their edges; the last has over 768 tiles
@pytest.mark.parametrize("nodes", [(7, 7, 7), (16, 8, 8), (17, 9, 13), (33, 15, 7), (97, 81, 65)])
@pytest.mark.parametrize("kind", ["narrow", "cell", "wide", "none"])
def test_iterates_follow_the_oracle(nodes, kind):
    s, N, rhs, n = _system(nodes, kind)
    if kind == "none":
        rhs = np.random.default_rng(8).standard_normal(n)
    r = torch.from_numpy(rhs).cuda()
    for m in (1, 2, 7):
        want, it, _ = ofd.jacobi_pcg(N, rhs, rtol=0.0, maxiter=m)
        got, info = s.solve(rtol=0.0, maxiter=m, rhs=r, check_every=5)
        assert info["iterations"] == m and not info["converged"]
        err = np.linalg.norm(got.cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= 1e-11, (nodes, kind, m, err)
        got, info = s.solve(rtol=0.0, maxiter=m, rhs=r, precision="fp32", inner_rtol=1e-30,
                            max_outer=1)
        err = np.linalg.norm(got.cpu().numpy() - want) / np.linalg.norm(want)
        own = np.linalg.norm(_pcg32(N, rhs, m) - want) / np.linalg.norm(want)
        assert info["iterations"] == m and err <= 30 * own + 1e-6, (nodes, kind, m, err, own)
    if n < 2000 and kind != "none":  # without rows only the ridge holds linear fields
        want, it, ok = ofd.jacobi_pcg(N, rhs, rtol=1e-8)
        got, info = s.solve(rtol=1e-8, rhs=r)
        # long runs on these random rows (condition ~1e7) lose orthogonality
        # at a rate that the order of the sums decides: counts within a tenth,
        # the residual below is the test
        assert ok and info["converged"] and abs(info["iterations"] - it) <= 0.1 * it + 2
        res = np.linalg.norm((rhs - N @ got.cpu().numpy()) / np.sqrt(N.diagonal()))
        assert res <= 1.1e-8 * np.linalg.norm(rhs / np.sqrt(N.diagonal()))
    s.close()


def test_rows_change_the_form():
    """One handle, rows of every width in turn; a zero right-hand side."""
    from loopstructural_amd import fd_system as fs

    s, _, _, n = _system((17, 9, 13), "none")
    c, info = s.solve(rtol=1e-8)
    assert info["converged"] and float(c.abs().max()) == 0.0
    for kind in ("cell", "wide", "narrow", "cell"):
        one, N, rhs, _ = _system((17, 9, 13), kind, seed=5)
        s.set_rows(one.rows)
        got, info = s.solve(rtol=1e-11)
        want = sparse.linalg.spsolve(N.tocsc(), rhs)
        assert info["converged"]
        assert np.linalg.norm(got.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)
        one.close()
    s.close()
