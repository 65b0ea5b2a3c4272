"""Tile heights up to the largest that the entry points accept: a height beyond
the grid is one chunk of all its rows, so the right-hand side, an adaptive run
with its step log, a batch and the adjoint's product give the bits of the height
equal to the grid's rows."""
import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


def _run(c, rows, batch):
    import sgnx
    s = sgnx.SGN2D(**c.solver_kwargs())
    s.set_rhs_kernel(1, rows)
    r = s.rhs(c.U0, 0.3)
    s.upload(c.U0)
    dt0 = s.cflTimeStep(None, 0.5)
    opts = sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=4)
    if batch:
        b = sgnx.Batch([s])
        st = b.integrateAdaptive(0.0, 1e9, [dt0], opts)[0]
        b.close()
        log = np.zeros(0)
    else:
        st, log = s.integrateAdaptive(0.0, 1e9, dt0, opts, step_log_cap=8)
        log = np.asarray(log).ravel()
    out = r, s.download(), log, st.as_dict()
    s.close()
    return out


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("Ny", [2, 6])
@pytest.mark.parametrize("rows", [2 ** 31 - 1, 2 ** 31 - 2, 2 ** 30])
def test_a_height_beyond_the_grid_is_the_grid(rows, Ny, batch):
    from sgnx import cases
    c = cases.gate(Nx=8, Ny=Ny)
    got, want = _run(c, rows, batch), _run(c, Ny, batch)
    for a, b, what in zip(got, want, ("rhs", "state", "log")):
        assert_bitwise(a, b, what)
    assert got[3] == want[3]


def test_products_at_the_largest_height(monkeypatch):
    import sgnx
    from sgnx import cases
    c = cases.gate(Nx=8, Ny=6)
    W = np.random.default_rng(2).normal(size=c.U0.size)
    got = []
    for rows in (6, 2 ** 31 - 1):
        monkeypatch.setenv("SGNX_VJP_ROWS", str(rows))
        s = sgnx.SGN2D(**c.solver_kwargs())
        s.setDepth(c.depth["Hnod"])
        got.append(s.rhs_vjp(c.U0, W, 0.3))
        s.close()
    for a, b, what in zip(got[0], got[1], ("Ubar", "thetaBar")):
        assert_bitwise(a, b, what)
