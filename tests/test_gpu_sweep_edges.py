"""The row sweep (variant 1) where its work split and its branch-free quotients
can go wrong: strips with one to five columns, chunks of one row, an odd number
of rows and a remainder, every side kind, and states with zeros of both signs,
subnormal, tiny and huge entries, depths with a significand of ones, infinities
and NaN. Finite states: the oracle's RHS bit for bit (a NaN or infinity that
overflow makes compares as such); others: the element-row tiles (variant 0)."""
import numpy as np
import pytest

import oracle_lib as OL

pytestmark = pytest.mark.gpu

SIDES = [("periodic",) * 4, ("periodic", "periodic", "wall", "wall"), ("wall",) * 4,
         ("inflow", "wall", "wall", "wall"), ("wall", "wall", "periodic", "periodic")]


def _case(Nx, Ny, bc, seed):
    from sgnx import cases
    Lx, Ly = 1.7 * Nx, 1.3 * Ny
    par = cases.Params(g=9.81, c=9.4, gamma=1.5)
    depth = cases.random_depth(4, Nx, Ny, Lx, Ly, seed, bc)
    inflow = cases.inflow_table(Ny, 4, 0.9, 1.5, 0.02) if bc[0] == "inflow" else None
    U0 = cases.random_state(Nx * Ny * 25, seed)
    return cases.Case("edges", 4, Nx, Ny, Lx, Ly, par, depth, bc, U0, inflow=inflow)


def _special(U, nd, seed, kind):
    U = U.copy()
    rng = np.random.default_rng(seed)
    mom = rng.permutation(np.arange(nd, 5 * nd))
    part = np.array_split(mom[:mom.size * 3 // 4], 6)
    U[part[0]] = 0.0
    U[part[1]] = -0.0
    if kind == "tiny":
        U[part[2]] *= 1e-310
        U[part[3]] *= 2.0 ** -899
        U[part[4]] *= 1e-160
        U[part[5]] = 5e-324
    elif kind == "huge":
        U[part[2]] *= 1e120
        U[part[3]] *= 1e240
        U[part[4]] *= 1e300
    h = rng.permutation(nd)[:nd // 8]
    U[h] = np.float64.fromhex("0x1.fffffffffffffp-1")
    if kind == "nonfinite":
        U[part[2][0]], U[part[3][0]], U[part[4][0]] = np.inf, -np.inf, np.nan
        U[h[0]], U[h[1]] = np.inf, np.nan
    return U


def _same(got, want, what):
    eq = (got.view(np.uint64) == want.view(np.uint64)) | (np.isnan(got) & np.isnan(want))
    assert eq.all(), f"{what}: {np.count_nonzero(~eq)} of {eq.size} entries differ"


@pytest.mark.parametrize("kind", ["tiny", "huge", "nonfinite"])
@pytest.mark.parametrize("Nx,Ny,sides,rows", [(2, 2, 0, 1), (6, 5, 1, 2), (7, 9, 2, 4),
                                              (13, 6, 3, 3), (9, 11, 4, 5), (10, 7, 3, 16)])
def test_sweep_edges(Nx, Ny, sides, rows, kind):
    import sgnx
    c = _case(Nx, Ny, SIDES[sides], 3 + Nx)
    U = _special(c.U0, c.nd, 11 * Nx + Ny, kind)
    s = sgnx.SGN2D(**c.solver_kwargs())
    try:
        s.set_rhs_kernel(0)
        want = s.rhs(U, 0.37)
        if kind != "nonfinite":
            o = OL.Oracle.from_case(c)
            want = o.rhs(U, 0.37)
            o.close()
        s.set_rhs_kernel(1, rows)
        _same(s.rhs(U, 0.37), want, f"{Nx}x{Ny} rows {rows} {kind}")
    finally:
        s.close()
