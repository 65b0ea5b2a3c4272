"""The product kernel of the adjoint where its work split can go wrong: strips
of one to five columns, chunks of one row, of an odd number, with a remainder
and of the whole grid, every side kind, with and without the still-depth part.
Reference: central differences of the oracle in random directions (error
O(eps^2) plus rounding 1e-16 / eps, so a relative 1e-6 as in the other adjoint
tests), and the heights among themselves bit for bit, since every sum has one
order whatever the split."""
import numpy as np
import pytest

from test_gpu_adjoint import EPS, TOL, _oracle, _rel, _state

pytestmark = pytest.mark.gpu

SIDES = [("periodic",) * 4, ("periodic", "periodic", "wall", "wall"), ("wall",) * 4,
         ("inflow", "wall", "wall", "wall"), ("wall", "wall", "periodic", "periodic")]


def _case(Nx, Ny, bc, seed):
    from sgnx import cases
    Lx, Ly = 1.7 * Nx, 1.3 * Ny
    par = cases.Params(g=9.81, c=9.4, gamma=1.5)
    depth = cases.random_depth(4, Nx, Ny, Lx, Ly, seed, bc)
    inflow = cases.inflow_table(Ny, 4, 0.9, 1.5, 0.02) if bc[0] == "inflow" else None
    return cases.Case("vjp-edges", 4, Nx, Ny, Lx, Ly, par, depth, bc,
                      cases.random_state(Nx * Ny * 25, seed), inflow=inflow)


@pytest.mark.parametrize("Nx,Ny,sides", [(2, 2, 0), (2, 3, 4), (4, 7, 1), (5, 2, 3), (6, 5, 2),
                                         (11, 9, 3), (13, 4, 0), (15, 34, 4), (24, 33, 2)])
def test_vjp_edges(Nx, Ny, sides, monkeypatch):
    import sgnx
    seed = 7 * Nx + Ny
    c = _case(Nx, Ny, SIDES[sides], seed)
    rng = np.random.default_rng(seed)
    theta = c.depth["Hnod"] + 0.01 * rng.uniform(-1, 1, c.nd)
    U = _state(c, seed)
    W = rng.normal(size=U.size)
    t = 0.37
    runs = []
    for rows in ("1", "2", "3", "16", "33", ""):
        if rows:
            monkeypatch.setenv("SGNX_SWEEP_ROWS", rows)
        else:
            monkeypatch.delenv("SGNX_SWEEP_ROWS")
        s = sgnx.SGN2D(**c.solver_kwargs())
        s.setDepth(theta)
        runs.append(s.rhs_vjp(U, W, t))
        s.close()
    Ub, thb = runs[0]
    for k, (u, th) in enumerate(runs[1:]):
        assert np.array_equal(u, Ub) and np.array_equal(th, thb), f"height {k}"
    o = _oracle(c, theta)
    dU = rng.uniform(-1.0, 1.0, U.size) * np.repeat([0.05, 0.05, 0.05, 0.02, 0.02], c.nd)
    for v in range(5):
        d = np.zeros_like(dU)
        d[v * c.nd:(v + 1) * c.nd] = dU[v * c.nd:(v + 1) * c.nd]
        fd = W @ (o.rhs(U + EPS * d, t) - o.rhs(U - EPS * d, t)) / (2 * EPS)
        assert _rel(Ub @ d, fd) < TOL, (v, Ub @ d, fd)
    dth = rng.uniform(-1.0, 1.0, c.nd) * 0.05
    fdt = W @ (_oracle(c, theta + EPS * dth).rhs(U, t) -
               _oracle(c, theta - EPS * dth).rhs(U, t)) / (2 * EPS)
    assert _rel(thb @ dth, fdt) < TOL, (thb @ dth, fdt)
